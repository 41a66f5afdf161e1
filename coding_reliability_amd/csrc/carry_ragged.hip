// Pair-distance histograms of codes whose word count is no power of two, by
// recursion over the carries (gfx950): the same raw[] as the pair kernel for
// short multipliers.
//
// The words i < N fall into aligned blocks, one of 2^m words for each 1 bit m of N.
// F_m(c, c')[d]: pairs (t, t') of m-bit numbers whose products leave the carries
// c, c' and differ in d of the m low places; from the low end,
//   F_{m+1}(d, d')[x] = sum over bits y, y' of F_m(c, c')[x - (y ^ y')],
//   c + A*b = 2 d + y, c' + A*b' = 2 d' + y'   (one c and b for each d and y),
// A odd.  The words 2^m s + t of block s of 2^m words are A*t plus A*s above the
// low m places, so two blocks s, s' differ in popcount((c + A*s) ^ (c' + A*s'))
// places there: the 1 bit m of N, whose block is s' = N >> m less one, pairs its
// block with the s' blocks below it and itself by counting E(c, c')[e], the s
// with e such places, and adding sum over c, c', d, e of F[d] * E[e] at d + e.
// The low bits of N below 2^T > A, where blocks are fewer words than carries, are
// a tail of up to 2^T - 1 words that ragged_tail pairs one by one.
//
// Bound by the latency of the levels and their launches (3 us each) for the
// smallest multipliers, by the products of E and F in LDS for the others.
// Measured for one call, A = 61: 65537 words 72 us (0.27 ms in the pair
// kernel), 262143 words 0.22 ms (3.7 ms), 1048575 words 0.32 ms (58.5 ms); A =
// 511, 1048575 words 2.6 ms, A = 1021 8.2 ms.
#include <algorithm>

#include "cr_device.h"
#include "cr_internal.h"

namespace cr {
namespace {

using namespace dev;

using u64 = unsigned long long;
constexpr uint32_t kMaxA = 1024;
constexpr uint32_t kMaxLevels = 20;   // of N < 2^21 words
constexpr uint32_t kLow = kMaxLevels + 1;   // distances of the low places
constexpr uint32_t kHigh = 32;        // of the places above: words below 2^31
constexpr uint32_t kTailRows = 4;     // rows a lane of ragged_tail

__global__ __launch_bounds__(256) void ragged_init(u64 *__restrict__ F, uint32_t states, const DirectResult out) {
    direct_start(out);
    const uint32_t s = blockIdx.x * 256 + threadIdx.x;
    if (s < states) F[s] = s == 0;
}

// F_{m+1} from F_m with nb distances: thread (state, distance blockIdx.y).
__global__ __launch_bounds__(256) void ragged_step(const u64 *__restrict__ in, u64 *__restrict__ out, uint32_t A,
                                                   uint32_t states, uint32_t nb) {
    const uint32_t s = blockIdx.x * 256 + threadIdx.x, x = blockIdx.y;
    if (s >= states) return;
    const uint32_t d = s / A, dd = s - d * A;
    auto before = [A](uint32_t v) { return v < A ? v : v - A; };
    const uint32_t r0 = before(2 * d) * A, r1 = before(2 * d + 1) * A, c0 = before(2 * dd), c1 = before(2 * dd + 1);
    u64 n = 0;
    if (x < nb) n = in[(uint64_t)x * states + r0 + c0] + in[(uint64_t)x * states + r1 + c1];
    if (x > 0) n += in[(uint64_t)(x - 1) * states + r0 + c1] + in[(uint64_t)(x - 1) * states + r1 + c0];
    out[(uint64_t)x * states + s] = n;
}

// Blocks s of a chunk of `share` below `last` against block `last`, and (the
// chunk after them) `last` against itself; a wave takes 64 carry pairs.  nb, eb: distances of the
// low places and of those above.
__global__ __launch_bounds__(64) void ragged_blocks(const u64 *__restrict__ F, uint32_t A, uint32_t states, uint32_t nb,
                                                    uint32_t eb, uint32_t last, uint32_t share,
                                                    uint32_t chunks, uint32_t nbins, const DirectResult out) {
    __shared__ uint32_t high[kHigh * kStride];
    __shared__ u64 sum[(kLow + kHigh) * kStride];
    const uint32_t lane = threadIdx.x, chunk = blockIdx.x % chunks, s = blockIdx.x / chunks * 64 + lane;
    for (uint32_t e = 0; e < kHigh; ++e) high[e * kStride + lane] = 0;
    for (uint32_t e = 0; e < kLow + kHigh; ++e) sum[e * kStride + lane] = 0;
    __syncthreads();
    const bool itself = chunk == chunks - 1;
    if (s < states) {
        const uint32_t c = s / A, w = s - c * A + A * last;
        const uint32_t first = itself ? last : chunk * share, end = itself ? last + 1 : min(first + share, last);
        uint32_t v = c + A * first;
        for (uint32_t b = first; b < end; ++b, v += A) lds_inc(high + __popc(v ^ w) * kStride + lane);
        const uint32_t weight = itself ? 1 : 2;  // ordered pairs
        for (uint32_t x = 0; x < nb; ++x) {
            const u64 f = F[(uint64_t)x * states + s] * weight;
            if (f == 0) continue;
            u64 *const at = sum + x * kStride + lane;
            for (uint32_t e = 0; e < eb; ++e) at[e * kStride] += f * high[e * kStride + lane];
        }
    }
    __syncthreads();
    u64 *const dst = hist_copy(out.copies, nbins, kHistCopies);
    for (uint32_t b = lane; b < nbins && b < kLow + kHigh; b += 64) {
        u64 n = 0;
        for (uint32_t l = 0; l < 64; ++l) n += sum[b * kStride + ((l + lane) & 63)];
        if (n) atomicAdd(dst + b, n);
    }
}

// The `tail` last words against all N, ordered: a pair with an earlier word
// counts twice.  A wave takes 64 kTailRows rows and, lanes sharing a column, all tail words.
__global__ __launch_bounds__(64) void ragged_tail(uint32_t A, uint32_t N, uint32_t tail, uint32_t nbins,
                                                  const DirectResult out) {
    extern __shared__ uint32_t lds[];  // counters of earlier rows, then of tail rows, a row for the others
    const uint32_t lane = threadIdx.x, start = N - tail;
    lds_clear(lds, 2 * nbins + 1);
    for (uint32_t r0 = blockIdx.x * 64 * kTailRows; tail && r0 < N; r0 += gridDim.x * 64 * kTailRows) {
        uint32_t w[kTailRows], *row[kTailRows];
#pragma unroll
        for (uint32_t r = 0; r < kTailRows; ++r) {
            const uint32_t i = r0 + r * 64 + lane;
            w[r] = A * i;
            row[r] = lds + lane + (i < start ? 0 : nbins) * kStride;
            if (i >= N) row[r] = nullptr;
        }
        uint32_t v = A * start;
        for (uint32_t j = 0; j < tail; ++j, v += A)
#pragma unroll
            for (uint32_t r = 0; r < kTailRows; ++r)
                lds_inc(row[r] ? row[r] + __popc(w[r] ^ v) * kStride : lds + 2 * nbins * kStride + lane);
    }
    __syncthreads();
    u64 *const dst = hist_copy(out.copies, nbins, kHistCopies);
    for (uint32_t b = lane; b < nbins; b += 64) {
        u64 n = 0;
        for (uint32_t l = 0; l < 64; ++l) {
            const uint32_t at = (l + lane) & 63;
            n += 2ull * lds[b * kStride + at] + lds[(nbins + b) * kStride + at];
        }
        if (n) atomicAdd(dst + b, n);
    }
    direct_finish(out, nbins, lds);
}

}  // namespace

// Blocks s that a wave counts: enough waves for the device, but at least as many
// blocks as its multiplications of E with F take time for (128 to 4096).
static uint32_t blocks_share(uint32_t states, uint32_t last) {
    uint32_t share = 128;
    while (share < 4096 && (uint64_t)share * 2048 * 64 < (uint64_t)states * last) share *= 2;
    return share;
}
static uint32_t high_bins(uint32_t A, uint32_t last) {
    const uint32_t most = A - 1 + A * last;
    return most ? 33 - (uint32_t)__builtin_clz(most) : 1;
}

bool carry_ragged_plan(uint64_t A, uint64_t num_words, CarryRaggedPlan *p) {
    if (A == 0 || num_words < 2 || num_words >> (kMaxLevels + 1)) return false;
    while ((A & 1) == 0) A >>= 1;  // an even multiplier has its odd part's distances
    if (A >= kMaxA) return false;
    p->A = (uint32_t)A;
    p->N = (uint32_t)num_words;
    // 2^T > A; a tail below 2^7 words costs less than the launches of its bits
    p->T = std::max(32 - (uint32_t)__builtin_clz((uint32_t)A), 7u);
    p->states = p->A * p->A;
    p->levels = 31 - (uint32_t)__builtin_clz(p->N);    // the highest bit of N
    if (p->levels < p->T) return false;
    p->nbins = 64 - (uint32_t)__builtin_clzll(A * (num_words - 1)) + 1;
    p->tail = p->N & ((1u << p->T) - 1);
    p->table_bytes = (uint64_t)p->states * (p->levels + 1) * sizeof(u64);
    // launches, 12 ps a counter of a level, 2 ps a product of E and F (measured 0.5
    // to 1.1 of this at A = 61 .. 1021 and 2^16 .. 2^20 words): the pair kernel keeps
    // codes below some 30000 words
    double s = 25e-6 + (double)p->tail * p->N / 8e12;
    for (uint32_t m = 0; m <= p->levels; ++m) {
        s += 3e-6 + 12e-12 * (double)p->states * (m + 1);
        if (m >= p->T && (p->N >> m & 1)) {
            const uint32_t last = (p->N >> m) - 1, share = blocks_share(p->states, last);
            s += 6e-6 + p->states * (last / 6e12 + ((last + share - 1) / share + 1.0) * (m + 1) *
                                                       high_bins(p->A, last) * 2e-12);
        }
    }
    p->seconds = s;
    return true;
}

cr_status carry_ragged_run(const CarryRaggedPlan &p, void *table0, void *table1, const DirectResult &out, int cus,
                           hipStream_t stream) {
    u64 *F = static_cast<u64 *>(table0), *next = static_cast<u64 *>(table1);
    const uint32_t wgs = (p.states + 255) / 256, waves = (p.states + 63) / 64;
    hipLaunchKernelGGL(ragged_init, dim3(wgs), dim3(256), 0, stream, F, p.states, out);
    CR_HIP(hipGetLastError());
    for (uint32_t m = 0;; ++m) {
        if (m >= p.T && (p.N >> m & 1)) {
            const uint32_t last = (p.N >> m) - 1, share = blocks_share(p.states, last);
            const uint32_t chunks = (last + share - 1) / share + 1, eb = high_bins(p.A, last);
            hipLaunchKernelGGL(ragged_blocks, dim3(waves * chunks), dim3(64), 0, stream, F, p.A, p.states, m + 1, eb, last,
                               share, chunks, p.nbins, out);
            CR_HIP(hipGetLastError());
        }
        if (m == p.levels) break;
        hipLaunchKernelGGL(ragged_step, dim3(wgs, m + 2), dim3(256), 0, stream, F, next, p.A, p.states, m + 1);
        CR_HIP(hipGetLastError());
        std::swap(F, next);
    }
    const uint32_t blocks = std::max(1u, std::min(p.tail ? (p.N + 64 * kTailRows - 1) / (64 * kTailRows) : 1u,
                                                  8u * (uint32_t)cus));
    hipLaunchKernelGGL(ragged_tail, dim3(blocks), dim3(64), (2 * p.nbins + 1) * kStride * sizeof(uint32_t), stream, p.A,
                       p.N, p.tail, p.nbins, out);
    CR_HIP(hipGetLastError());
    return CR_OK;
}

}  // namespace cr
