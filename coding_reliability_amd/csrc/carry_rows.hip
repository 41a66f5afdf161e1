// One-dimensional grid histograms by recursion over the carries of the product
// (gfx950): hist[d] = #{(i, s) : i < 2^n, popcount(A*i ^ v_s) = d} for a list of
// samples v_s, the quantity the rectangle kernel counts pair by pair.
//
// Against one sample v, the words A*i (A odd) whose low parts leave the same
// carry c < A are alike from there on.  With G_r(c)[d] the number of ways to
// choose the top r bits of i so that what follows c differs from v in d places,
//   G_0(c)[d] = [popcount(c ^ (v >> n)) = d],
//   G_{r+1}(c)[d] = G_r(c >> 1)[d - e] + G_r((c + A) >> 1)[d - 1 + e],
//   e = (c & 1) ^ bit n - 1 - r of v,
// and G_n(0) is the sample's histogram: A * n * (n + 1) counters instead of
// 2^n words.  An even A = 2^z * a has the words of a above z zero bits.
//
// A workgroup holds one sample's G in LDS, [distance][carry] with a thread per
// carry (consecutive lanes read consecutive or equal carries: no bank
// conflicts), and updates it in place from the largest distance down, kBins
// distances at a time: distance d reads only d and d - 1.  Up to 64 carries a
// sample takes one wave, without barriers, and a workgroup four samples.  Bound
// by LDS, two reads and a write per counter, and for few samples by the chain
// of n levels.  Measured: a call with a 6-bit A, n = 32 and 1001 samples 43 us,
// against 449 ms in the rectangle kernel (4.3e12 pairs at one LDS increment
// each).
#include <algorithm>
#include <cmath>

#include "cr_device.h"
#include "cr_internal.h"

namespace cr {
namespace {

using namespace dev;

constexpr int kBins = 8;                   // distances per in-place step
constexpr uint32_t kWaves = 4;             // samples of a workgroup of one wave each
constexpr uint32_t kLdsBytes = 150 << 10;  // of the 160 KB of a CU

// rows: a multiple of kBins above every distance; counters of distances no
// level has reached yet are zero.
template <class T, bool WAVE>
__global__ __launch_bounds__(WAVE ? 64 * kWaves : 1024) void carry_rows(uint32_t A, uint32_t z, uint32_t n,
                                                   const uint64_t *__restrict__ cols, uint32_t ncols, uint32_t rows,
                                                   uint32_t nbins, const DirectResult out) {
    extern __shared__ unsigned char lds_raw[];
    direct_start(out);
    const uint32_t wave = WAVE ? threadIdx.x / 64 : 0, c = threadIdx.x - 64 * wave, P = WAVE ? 64 : blockDim.x;
    T *const G = reinterpret_cast<T *>(lds_raw) + wave * rows * 64;
    // a wave's LDS accesses execute in order
    auto sync = [] {
        if (WAVE)
            __builtin_amdgcn_wave_barrier();
        else
            __syncthreads();
    };
    const bool act = c < A;
    const uint32_t c0 = act ? c >> 1 : 0, c1 = act ? (c + A) >> 1 : 0;
    const uint32_t maxc = A - 1;
    unsigned long long acc = 0;  // thread b < 64: distance b over this workgroup's samples
    const uint32_t per = WAVE ? kWaves : 1;
    for (uint32_t q = blockIdx.x * per + wave; q < ncols; q += gridDim.x * per) {
        const uint64_t full = cols[q], v = full >> z;
        const uint32_t below = (uint32_t)__popcll(full & ((1ull << z) - 1));
        const uint64_t top = v >> n;
        // distances a level can have: those of the carries, and one more a level
        const uint64_t span = top | maxc;
        const uint32_t w0 = span ? 64 - (uint32_t)__clzll(span) : 0;
        for (uint32_t b = 0; b < rows; ++b) G[b * P + c] = 0;
        if (act) G[(uint32_t)__popcll((uint64_t)c ^ top) * P + c] = 1;
        sync();
        for (uint32_t r = 0; r < n; ++r) {
            const uint32_t bit = (uint32_t)(v >> (n - 1 - r)) & 1;
            const bool e = ((c & 1) ^ bit) != 0;
            const T *const same = G + (e ? c1 : c0), *const next = G + (e ? c0 : c1);
            const uint32_t blocks = (w0 + r + 1) / kBins + 1;  // distances 0 .. w0 + r + 1
            for (uint32_t k = blocks; k-- > 0;) {
                const uint32_t b0 = k * kBins;
                T x[kBins];
#pragma unroll
                for (int u = 0; u < kBins; ++u) {
                    x[u] = same[(b0 + u) * P];
                    if (u > 0 || b0 > 0) x[u] += next[(b0 + u - 1) * P];
                }
                sync();
                if (act) {
#pragma unroll
                    for (int u = 0; u < kBins; ++u) G[(b0 + u) * P + c] = x[u];
                }
            }
            sync();
        }
        if (c < nbins && c >= below) acc += G[(c - below) * P];
        sync();
    }
    __syncthreads();
    if (c < nbins && acc) atomicAdd(hist_copy(out.copies, nbins, kHistCopies) + c, acc);
    direct_finish(out, nbins, reinterpret_cast<uint32_t *>(lds_raw));
}

}  // namespace

bool carry_rows_plan(uint64_t A, uint32_t n, uint64_t ncols, uint32_t nbins, CarryRowsPlan *p) {
    if (A == 0 || n == 0 || n > 48 || ncols >> 32 || nbins > 64) return false;
    p->z = (uint32_t)__builtin_ctzll(A);
    const uint64_t a = A >> p->z;
    if (a > 1024) return false;
    p->A = (uint32_t)a;
    p->n = n;
    // a sample's counts sum to 2^n, and no distance holds all of them when n
    // = 32 (the low n bits run over every residue, the rest spans 10 bits)
    p->wide = n > 32;
    // counters up to distance 64 of the widest words, written in blocks
    p->rows = (nbins + 1 + kBins - 1) / kBins * kBins;
    p->threads = (std::max(p->A, 64u) + 63) & ~63u;
    p->lds = (size_t)p->rows * p->threads * (p->wide ? 8 : 4);
    if (p->lds > kLdsBytes) return false;
    // LDS time of the counters (three accesses each, 128 bytes a clock and CU,
    // about half of it reached) against the rectangle kernel's 9.5e12 pairs/s
    const double counters = (double)p->threads * n * (0.5 * n + 12);
    const double recursion = counters * (p->wide ? 24 : 12) / (256 * 128 * 2.4e9 * 0.5);
    return recursion < std::ldexp(1.0, (int)n) / 9.5e12;
}

cr_status launch_carry_rows(const CarryRowsPlan &p, const uint64_t *cols, uint32_t ncols, uint32_t nbins,
                            const DirectResult &out, int cus, hipStream_t stream) {
    const bool wave = p.threads == 64;
    const void *k = wave ? (p.wide ? reinterpret_cast<const void *>(&carry_rows<unsigned long long, true>)
                                   : reinterpret_cast<const void *>(&carry_rows<uint32_t, true>))
                         : (p.wide ? reinterpret_cast<const void *>(&carry_rows<unsigned long long, false>)
                                   : reinterpret_cast<const void *>(&carry_rows<uint32_t, false>));
    const uint32_t per = wave ? kWaves : 1, threads = p.threads * per;
    const size_t lds = p.lds * per;
    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k, (int)threads, lds) != hipSuccess || per_cu <= 0)
        return fail(CR_ERR_DEVICE, "occupancy query failed for the carry rows kernel");
    const uint32_t blocks = std::min<uint32_t>((ncols + per - 1) / per, (uint32_t)per_cu * (uint32_t)cus);
    uint32_t a_A = p.A, a_z = p.z, a_n = p.n, a_nc = ncols, a_rows = p.rows, a_nb = nbins;
    void *args[] = {&a_A, &a_z, &a_n, (void *)&cols, &a_nc, &a_rows, &a_nb, (void *)&out};
    CR_HIP(hipLaunchKernel(k, dim3(blocks), dim3(threads), args, lds, stream));
    return CR_OK;
}

}  // namespace cr
