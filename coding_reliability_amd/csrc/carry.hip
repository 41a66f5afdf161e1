// Exhaustive AN distance distributions by recursion over the carries of the
// product (gfx950): the same raw[] as the pair kernel for 2^k words of a short
// multiplier, without visiting pairs.
//
// Bit by bit from the low end, A*i (A odd) leaves a carry c < A: with the next
// bit b of i the word's next bit is (c + A*b) & 1 and the carry (c + A*b) >> 1.
// For two words with carries c and c', let Q_r(c, c')[d] be the number of ways
// to choose r more bits for each so that what follows differs in d places:
//   Q_0(c, c')[d] = [popcount(c ^ c') = d],
//   Q_{r+f}(c, c')[d] = sum over i, j < 2^f of
//                       Q_r((c + A*i) >> f, (c' + A*j) >> f)[d - popcount(y ^ y')],
//   y = (c + A*i) mod 2^f, y' = (c' + A*j) mod 2^f,
// and Q_k(0, 0) is the distribution over ordered pairs.  The A^2 carry pairs
// times at most n + 1 distances replace the 2^(2k) pairs of words: with
// A = 61 and k = 32 some 2^22 counters a level instead of 2^38 transformed
// elements.
//
// Three kernels, tables in the layout [distance][c * A + c'] (lanes run over
// c', so a load is a few contiguous runs):
//   carry_init   Q_r0 from the words themselves, r0 = 4 (a workgroup's 64
//                carry pairs, 256 pairs of words each, counted in LDS)
//   carry_step   f = 2 (once f = 1 for an odd number of levels): a thread per
//                counter, 16 loads
//   carry_final  Q_k(0, 0): the last T levels at once, 2^T > A: every pair of
//                T-bit low parts looks up its carries
// The tables of short multipliers stay in the L2s, so a level costs its launch
// and the latency of one round of loads (3.2 us for two levels at A = 61, 4.6 in
// 64 bits, so steps take two levels, not one); longer ones are bound by the 16
// loads per counter (9 TB/s from L1 and L2 at A = 1021).  Measured for one
// call, against the spectral path that served these codes before: 6-bit A at
// k = 24 40 us (1.13 ms), at k = 32 57 us (993 ms), A = 1021 at k = 24 0.84 ms
// (14.9 ms).
#include <algorithm>
#include <vector>

#include "cr_device.h"
#include "cr_internal.h"

namespace cr {
namespace {

using namespace dev;

constexpr uint32_t kInitBits = 4;    // levels that carry_init takes at once
constexpr uint32_t kInitRows = 17;   // distances of Q_4: 4 + 12 + 1 at most
constexpr uint64_t kMaxTable = 1ull << 31;
constexpr uint32_t kFinalBins = 64;  // largest number of distances
constexpr uint32_t kGroup = 4;       // distances of a wave of carry_final
constexpr uint32_t kWaves = 8;       // waves of its workgroup
constexpr uint32_t kFinalRows = kGroup + 12;  // and the T <= 12 bits that shift them: 16

// Q_{kInitBits} for 64 carry pairs a workgroup, a quarter of the pairs of words a
// wave (6 levels at once were bound by the LDS of the few workgroups: 11 us for
// 3.4 and a step of 3.2).
__global__ __launch_bounds__(256) void carry_init(uint32_t *__restrict__ T, uint32_t A, uint32_t states, uint32_t nb,
                                                  const DirectResult out) {
    __shared__ uint32_t lds[kInitRows * kStride];
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    direct_start(out);
    for (uint32_t e = threadIdx.x; e < kInitRows * kStride; e += 256) lds[e] = 0;
    __syncthreads();
    const uint32_t s = blockIdx.x * 64 + lane;
    const uint32_t c = s / A, cc = s - c * A;
    if (s < states) {
        for (uint32_t i = wave * 4; i < wave * 4 + 4; ++i) {
            const uint32_t w = c + A * i;
#pragma unroll
            for (uint32_t j = 0; j < (1u << kInitBits); ++j) {
                const uint32_t d = __popc(w ^ (cc + A * j));
                lds_inc(lds + d * kStride + lane);
            }
        }
    }
    __syncthreads();
    if (s >= states) return;
    for (uint32_t b = wave; b < nb; b += 4) T[(uint64_t)b * states + s] = lds[b * kStride + lane];
}

// F levels: thread (s, blockIdx.y) computes distance blockIdx.y of carry pair s
// (several a thread measured slower up to A = 127, by a third at 61, and no
// faster beyond).  The source for low bits y, y' is popcount(y ^ y') distances
// below.
template <int F, class In, class Out>
__global__ __launch_bounds__(256) void carry_step(const In *__restrict__ Q, Out *__restrict__ T, uint32_t A,
                                                  uint32_t Ainv, uint32_t states, uint32_t nb_in) {
    const uint32_t s = blockIdx.x * 256 + threadIdx.x;
    if (s >= states) return;
    constexpr uint32_t M = (1u << F) - 1;
    const uint32_t c = s / A, cc = s - c * A, b = blockIdx.y;
    uint32_t row[M + 1], col[M + 1];  // next carry for low bits y
#pragma unroll
    for (uint32_t y = 0; y <= M; ++y) {
        row[y] = ((c + A * (((y - c) * Ainv) & M)) >> F) * A;
        col[y] = (cc + A * (((y - cc) * Ainv) & M)) >> F;
    }
    Out a = 0;
#pragma unroll
    for (uint32_t e = 0; e <= F; ++e) {
        const bool in = b - e < nb_in;  // wraps below 0
        const In *q = Q + (uint64_t)(in ? b - e : 0) * states;
        Out part = 0;
#pragma unroll
        for (uint32_t y = 0; y <= M; ++y)
#pragma unroll
            for (uint32_t z = 0; z <= M; ++z)
                if (__builtin_popcount(y ^ z) == e) part += (Out)q[row[y] + col[z]];
        a += in ? part : (Out)0;
    }
    T[(uint64_t)b * states + s] = a;
}

// Ordered-pair distribution: every pair (y, y') of T-bit low parts, y <= y'
// (counted twice when y < y'), adds Q(c(y), c(y')) shifted by popcount(y ^
// y').  Lanes run over y'; a wave takes kGroup distances of Q, each lane with a
// column of 64-bit counters in LDS.  The waves of a workgroup take the groups of
// one tile: the last workgroup's threads share the sum over the copies, which
// took a single wave 8 us.
template <class In>
__global__ __launch_bounds__(64 * kWaves) void carry_final(const In *__restrict__ Q, uint32_t A, uint32_t Ainv,
                                                           uint32_t T, uint32_t states, uint32_t nb, uint32_t nbins,
                                                           const DirectResult out) {
    __shared__ uint32_t flag;
    __shared__ unsigned long long counts[kWaves][kFinalRows * kStride];
    const uint32_t lane = threadIdx.x & 63, wave = uniform32(threadIdx.x >> 6);
    const uint32_t parts = (nb + kGroup * kWaves - 1) / (kGroup * kWaves);
    const uint32_t b0 = (blockIdx.x % parts * kWaves + wave) * kGroup;
    unsigned long long *const lds = counts[wave];
    for (uint32_t b = 0; b < kFinalRows; ++b) lds[b * kStride + lane] = 0;
    const uint32_t N = 1u << T, M = N - 1;
    const uint32_t cols = (N + 63) / 64;
    if (b0 < nb) {
        for (uint32_t t = blockIdx.x / parts; t < N * cols; t += gridDim.x / parts) {
            const uint32_t y = t / cols, z = (t - y * cols) * 64 + lane;
            if (z >= N || z < y) continue;
            // A * i < 2^(2T) <= 2^24
            const uint32_t c = (A * ((y * Ainv) & M)) >> T, cc = (A * ((z * Ainv) & M)) >> T;
            const In *q = Q + (uint64_t)b0 * states + c * A + cc;
            unsigned long long *const at = lds + __popc(y ^ z) * kStride + lane;
            const uint32_t w = z == y ? 0 : 1;
            unsigned long long v[kGroup];
#pragma unroll
            for (uint32_t b = 0; b < kGroup; ++b)
                v[b] = b0 + b < nb ? (unsigned long long)q[(uint64_t)b * states] << w : 0;
#pragma unroll
            for (uint32_t b = 0; b < kGroup; ++b) at[b * kStride] += v[b];
        }
        // four lanes a row, 16 columns each, in an order that spreads the banks
        const uint32_t row = lane / 4, part = lane & 3;
        unsigned long long s = 0;
        for (uint32_t l = 0; l < 16; ++l) s += lds[row * kStride + part * 16 + ((l + row) & 15)];
        s += __shfl_xor(s, 1, 64);
        s += __shfl_xor(s, 2, 64);
        if (part == 0 && b0 + row < nbins && s)
            atomicAdd(hist_copy(out.copies, nbins, kHistCopies) + b0 + row, s);
    }
    direct_finish(out, nbins, &flag);
}

template <int F, class In, class Out>
void launch_step(const void *Q, void *T, const CarryPlan &p, uint32_t nb_in, hipStream_t stream) {
    const dim3 grid((p.states + 255) / 256, nb_in + F);
    hipLaunchKernelGGL((carry_step<F, In, Out>), grid, dim3(256), 0, stream, (const In *)Q, (Out *)T, p.A, p.Ainv,
                       p.states, nb_in);
}

template <int F>
void launch_step_types(const void *Q, void *T, const CarryPlan &p, bool in64, bool out64, uint32_t nb_in,
                       hipStream_t stream) {
    if (in64)
        launch_step<F, unsigned long long, unsigned long long>(Q, T, p, nb_in, stream);
    else if (out64)
        launch_step<F, uint32_t, unsigned long long>(Q, T, p, nb_in, stream);
    else
        launch_step<F, uint32_t, uint32_t>(Q, T, p, nb_in, stream);
}

// Counters of Q_r sum to 4^r: 32 bits hold them up to r = 15.
bool wide(uint32_t r) { return r >= 16; }

}  // namespace

bool carry_plan(uint64_t A, uint32_t k, CarryPlan *p) {
    if (A == 0 || k > 32) return false;
    while ((A & 1) == 0) A >>= 1;  // an even multiplier has its odd part's distances
    if (A >= 4096) return false;
    p->A = (uint32_t)A;
    p->k = k;
    p->T = 32 - (uint32_t)__builtin_clz((uint32_t)A);         // 2^T > A
    p->hb = A > 1 ? 32 - (uint32_t)__builtin_clz((uint32_t)A - 1) : 0;  // bits of the largest carry
    if (k < p->T + kInitBits) return false;
    p->levels = k - p->T;
    p->states = p->A * p->A;
    uint32_t x = p->A;  // inverse modulo 2^32, correct to 3 bits, doubled by each Newton step
    for (int i = 0; i < 5; ++i) x *= 2u - p->A * x;
    p->Ainv = x;
    p->nbins = k + p->hb + 1;
    if (p->nbins > kFinalBins) return false;
    const uint64_t nb = p->levels + p->hb + 1;
    p->table_bytes = (uint64_t)p->states * nb * (wide(p->levels) ? 8 : 4);
    // Host and launch time of a call, then measured kernel rates (A = 61, 511 and
    // 1021, k = 14 .. 32): 100 ps a carry pair for the first and the last
    // kernel, two levels 3.2 us and 6.5 ps a counter in 32 bits, 4.4 us and 11 ps
    // in 64.
    double s = 17e-6 + 1.0e-10 * p->states;
    for (uint32_t r = kInitBits; r < p->levels;) {
        r += ((p->levels - r) & 1) ? 1 : 2;
        s += wide(r) ? 4.4e-6 : 3.2e-6;
        s += (wide(r) ? 11e-12 : 6.5e-12) * (double)p->states * (r + p->hb + 1);
    }
    p->seconds = s;
    return p->table_bytes <= kMaxTable;
}

cr_status carry_run(const CarryPlan &p, void *table0, void *table1, const DirectResult &out, int cus,
                    hipStream_t stream) {
    uint32_t r = kInitBits, nb = kInitBits + p.hb + 1;
    if (nb > kInitRows) return fail(CR_ERR_DEVICE, "carry recursion: %u distances", nb);
    hipLaunchKernelGGL(carry_init, dim3((p.states + 63) / 64), dim3(256), 0, stream, (uint32_t *)table0, p.A, p.states,
                       nb, out);
    CR_HIP(hipGetLastError());
    void *Q = table0, *T = table1;
    while (r < p.levels) {
        const uint32_t f = ((p.levels - r) & 1) ? 1 : 2;
        if (f == 1)
            launch_step_types<1>(Q, T, p, wide(r), wide(r + f), nb, stream);
        else
            launch_step_types<2>(Q, T, p, wide(r), wide(r + f), nb, stream);
        CR_HIP(hipGetLastError());
        std::swap(Q, T);
        r += f;
        nb += f;
    }
    const uint64_t tiles = ((uint64_t)1 << p.T) * (((1u << p.T) + 63) / 64);
    const dim3 blocks((uint32_t)std::min<uint64_t>(tiles, 2ull * cus) * ((nb + kGroup * kWaves - 1) / (kGroup * kWaves)));
    if (wide(r))
        hipLaunchKernelGGL(carry_final<unsigned long long>, blocks, dim3(64 * kWaves), 0, stream,
                           (const unsigned long long *)Q, p.A, p.Ainv, p.T, p.states, nb, p.nbins, out);
    else
        hipLaunchKernelGGL(carry_final<uint32_t>, blocks, dim3(64 * kWaves), 0, stream, (const uint32_t *)Q, p.A, p.Ainv,
                           p.T, p.states, nb, p.nbins, out);
    CR_HIP(hipGetLastError());
    return CR_OK;
}

cr_status ordered_finish(uint64_t words, uint32_t bins, const uint64_t *hist, uint64_t *raw, uint32_t nbins) {
    uint64_t total = 0;
    for (uint32_t b = 0; b < nbins; ++b) raw[b] = 0;
    for (uint32_t b = 0; b < bins; ++b) {
        total += hist[b];
        if (b == 0 ? hist[b] != words : b >= nbins ? hist[b] != 0 : (hist[b] & 1) != 0)
            return fail(CR_ERR_DEVICE, "carry recursion: inconsistent count at distance %u", b);
        if (b > 0 && b < nbins) raw[b] = hist[b] / 2;
    }
    if (total != words * words) return fail(CR_ERR_DEVICE, "carry recursion: inconsistent total");
    return CR_OK;
}

cr_status carry_finish(uint32_t k, uint32_t bins, const uint64_t *hist, uint32_t copies, uint64_t *raw,
                       uint32_t nbins) {
    const uint64_t stride = hist_copy_stride(bins);
    unsigned __int128 total = 0;
    for (uint32_t b = 0; b < nbins; ++b) raw[b] = 0;
    for (uint32_t b = 0; b < bins; ++b) {
        uint64_t s = 0;
        for (uint32_t c = 0; c < copies; ++c) s += hist[c * stride + b];
        total += s;
        if (b == 0) {
            if (s != 1ull << k) return fail(CR_ERR_DEVICE, "carry recursion: %llu words at distance 0", (unsigned long long)s);
        } else if (b >= nbins ? s != 0 : (s & 1) != 0) {
            return fail(CR_ERR_DEVICE, "carry recursion: inconsistent count at distance %u", b);
        } else if (b < nbins) {
            raw[b] = s / 2;
        }
    }
    if (total != (unsigned __int128)1 << (2 * k)) return fail(CR_ERR_DEVICE, "carry recursion: inconsistent total");
    return CR_OK;
}

}  // namespace cr
