// The recursion over carries (carry.hip) for long multipliers, tiled (gfx950).
//
// For a 16-bit A the tables of all A^2 carry pairs would be 100 GB a level and
// be written and read at every level.  A level of the recursion,
//   Q_{r+1}(c, c') = sum over bits b, b' of
//                    z^((c + b + c' + b') & 1) Q_r((c + A*b) >> 1, (c' + A*b') >> 1)
// (polynomials in z, the distance; A odd), takes a run of w carries to two runs
// of w/2 + 1: a tile of 32 x 32 carry pairs needs 2 x 2 tiles of 17 x 17 a level
// below, 4 x 4 of 9 x 9, 8 x 8 of 5 x 5, 16 x 16 of 3 x 3.  So two kernels take
// four levels each with the levels between in LDS, block by block of kSide x
// kSide carry pairs of the last level; the table between them (level 4, a block
// at a time, 100 MB) stays in the last-level cache:
//   tiles_low   level 4 of the carry pairs that the block comes from, 32 x 32
//               at a time: level 1 from the words themselves, levels 2, 3 in
//               LDS, four 8-bit counters a dword;
//   tiles_high  levels 5 .. 4 + F in LDS, two 16-bit counters a dword, and the
//               last one straight into the histogram: carry pair (c, c') serves
//               every pair (i, j) of low parts with those carries, shifted by
//               the distance of the low parts' own bits.
// A level-r polynomial sums to 4^r: 256 at level 4, 65536 at level 8, one more
// than the packed counters hold.  No coefficient takes the whole sum: for no odd
// A < 2^16 and no two carries are all 256 pairs of level 4 at one distance
// (enumerated; all c + A*i, i < 16, would have one parity, which leaves 112970
// carries of all A together), so neither are the 65536 of level 8, whose terms
// these are.
// By symmetry only blocks and tiles with c-tile <= c'-tile run; a tile off the
// diagonal counts twice.
//
// Two rows 2t, 2t + 1 of a run have three rows below: with s the parity of the
// run's first carry, row t of the run of bit s (N) serves both, rows t and t +
// 1 of the other run (S0, S1) one each; N adds the bit of the row's own parity,
// S the other.  So four outputs take 9 polynomials, not 16: LDS traffic is the
// largest part of both kernels (tiles_low: 3.9 of its 7.7 kilocycles a tile and
// CU, tiles_high<4>: 7 of 24 without bank conflicts; the rest is latency
// between barriers, one workgroup filling a CU's LDS).  Measured for one call
// with A = 58659: k = 24 88 ms, where the spectral path took 910 ms (2^40
// transformed elements); k = 20 37 ms (54 ms in the spectral path).
#include <algorithm>
#include <cmath>

#include "cr_device.h"
#include "cr_internal.h"

namespace cr {
namespace {

using namespace dev;

constexpr uint32_t kTile = 32;
constexpr uint32_t kGrid = 2048;  // level-4 carries a block comes from, each way
constexpr uint32_t kSide = 2016;  // carries of a block at the last level: kSide / 2^F + 1 <= kGrid / 2^F
constexpr uint32_t kLow = 4;      // levels of tiles_low
constexpr uint32_t kMaxLows = 65536 / kTile + 2;
static_assert(kSide % kTile == 0, "tiles start at multiples of kTile");
constexpr uint32_t kRows = 44;    // distances of a histogram in LDS

// Carries of a run l levels below a tile, and of all its 2^l runs.
constexpr uint32_t run_len(int l) { return l == 0 ? 32 : l == 1 ? 17 : l == 2 ? 9 : l == 3 ? 5 : 3; }
constexpr uint32_t run_all(int l) { return run_len(l) << l; }
constexpr uint32_t run_pairs(int l) { return (run_len(l) + 1) / 2; }

// Parities of the first carries of the 2^l runs l levels below a tile (bit p:
// run p), s being the tile's first carry.
template <int l>
__device__ __forceinline__ uint32_t run_parities(uint32_t s, uint32_t A) {
    uint32_t m = 0;
#pragma unroll
    for (uint32_t p = 0; p < (1u << l); ++p) m |= (((s + A * p) >> l) & 1) << p;
    return m;
}

// Rows N, S0, S1 below the row pair t of run p, l levels below a tile: indices
// into the runs one level further down; an S1 that no row uses may lie one
// past the last and is clamped.
struct Below {
    uint32_t n, s0, s1;
};
template <int l>
__device__ __forceinline__ Below below(uint32_t parities, uint32_t p, uint32_t t) {
    constexpr uint32_t other = run_len(l + 1) << l;  // from run p to run p + 2^l
    const uint32_t odd = ((parities >> p) & 1) * other;
    const uint32_t base = p * run_len(l + 1) + t;
    Below r;
    r.n = base + odd;
    r.s0 = base + other - odd;
    r.s1 = min(r.s0 + 1, run_all(l + 1) - 1);
    return r;
}

// 9 sources of one dword index into the sums of a quad's four outputs: zero
// (distance kept) and one (distance + 1).
__device__ __forceinline__ void quad_sums(const uint32_t (&x)[3][3], uint32_t (&zero)[4], uint32_t (&one)[4]) {
    one[0] = x[0][1] + x[1][0];
    one[1] = x[0][0] + x[1][2];
    one[2] = x[0][0] + x[2][1];
    one[3] = x[0][2] + x[2][0];
    zero[0] = x[0][0] + x[1][1];
    zero[1] = x[0][2] + x[1][0];
    zero[2] = x[0][1] + x[2][0];
    zero[3] = x[0][0] + x[2][2];
}

// --- levels 1 .. 4 -----------------------------------------------------------
constexpr uint32_t kLowThreads = 512;
constexpr int kLowDwords = 5;  // 20 distances: 3 + 16 + 1 at level 3

// Row pitch of a level's buffer: 32 consecutive quads read the end of one row
// of quads and the start of the next, which fall on different banks when the
// pitch is the quads of a row modulo 32.
constexpr uint32_t low_pitch(int l) { return (run_pairs(l - 1) << (l - 1)) + 32; }

// The four outputs of a quad of 8-bit polynomials, NOUT = 5 or 6 dwords (a
// polynomial times z moves its counters up a byte).
template <int l, int NOUT>
__device__ __forceinline__ void low_quad(const uint32_t *src, const Below &r, const Below &c,
                                         uint32_t (&o)[4][NOUT]) {
    constexpr uint32_t P = low_pitch(l + 1), S = run_all(l + 1) * P;
    const uint32_t rows[3] = {r.n * P, r.s0 * P, r.s1 * P}, cols[3] = {c.n, c.s0, c.s1};
    uint32_t prev[4] = {0, 0, 0, 0};
#pragma unroll
    for (int w = 0; w < NOUT; ++w) {
        uint32_t x[3][3];
#pragma unroll
        for (int a = 0; a < 3; ++a)
#pragma unroll
            for (int b = 0; b < 3; ++b) x[a][b] = w < kLowDwords ? src[w * S + rows[a] + cols[b]] : 0;
        uint32_t zero[4], one[4];
        quad_sums(x, zero, one);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            o[q][w] = zero[q] + __builtin_amdgcn_alignbit(one[q], prev[q], 24);
            prev[q] = one[q];
        }
    }
}

template <int l>
__device__ __forceinline__ void low_level(const uint32_t *src, uint32_t *dst, uint32_t rpar, uint32_t cpar) {
    constexpr uint32_t P = run_pairs(l), RP = P << l, D = low_pitch(l), S = run_all(l) * D;
    for (uint32_t q = threadIdx.x; q < RP * RP; q += kLowThreads) {
        const uint32_t rp = q / RP, cp = q - rp * RP;
        const uint32_t pr = rp / P, tr = rp - pr * P, pc = cp / P, tc = cp - pc * P;
        uint32_t o[4][kLowDwords];
        low_quad<l, kLowDwords>(src, below<l>(rpar, pr, tr), below<l>(cpar, pc, tc), o);
        const uint32_t at = (pr * run_len(l) + 2 * tr) * D + pc * run_len(l) + 2 * tc;
        const bool r1 = 2 * tr + 1 < run_len(l), c1 = 2 * tc + 1 < run_len(l);
#pragma unroll
        for (int w = 0; w < kLowDwords; ++w) {
            uint32_t *d = dst + w * S + at;
            d[0] = o[0][w];
            if (c1) d[1] = o[1][w];
            if (r1) d[D] = o[2][w];
            if (r1 && c1) d[D + 1] = o[3][w];
        }
    }
}

// Workgroup (col tile, row tile) of the kGrid x kGrid level-4 pairs: grid row
// p * (kGrid >> F) + t is carry ((R0 + A * p) >> F) + t.  V holds 24 bytes a
// pair: dword x the counters of distances 2x, 2x + 1, 2x + 12, 2x + 13, which
// tiles_high widens to pairs (2x, 2x + 12) and (2x + 1, 2x + 13) with a mask.
__global__ __launch_bounds__(kLowThreads) void tiles_low(uint4 *__restrict__ V, uint32_t A, uint32_t R0, uint32_t C0,
                                                         uint32_t F, uint32_t rows_used, uint32_t cols_used) {
    __shared__ uint32_t buf1[kLowDwords * run_all(3) * low_pitch(3)];  // level 1, then level 3
    __shared__ uint32_t buf2[kLowDwords * run_all(2) * low_pitch(2)];  // level 2
    const uint32_t W = kGrid >> F;
    const uint32_t r = blockIdx.y * kTile, c = blockIdx.x * kTile;
    const uint32_t pr = r / W, tr = r - pr * W, pc = c / W, tc = c - pc * W;
    if (tr >= rows_used || tc >= cols_used) return;
    const uint32_t sr = ((R0 + A * pr) >> F) + tr, sc = ((C0 + A * pc) >> F) + tc;
    {
        constexpr uint32_t D = run_all(3), S = D * low_pitch(3);
        for (uint32_t q = threadIdx.x; q < D * D; q += kLowThreads) {
            const uint32_t i = q / D, j = q - i * D;
            uint32_t *const at = buf1 + i * low_pitch(3) + j;
            const uint32_t pi = i / run_len(3), pj = j / run_len(3);
            const uint32_t v = ((sr + A * pi) >> 3) + i - pi * run_len(3);
            const uint32_t w = ((sc + A * pj) >> 3) + j - pj * run_len(3);
#pragma unroll
            for (int x = 0; x < kLowDwords; ++x) at[x * S] = 0;
#pragma unroll
            for (uint32_t b = 0; b < 4; ++b) {
                const uint32_t d = __popc((v + A * (b & 1)) ^ (w + A * (b >> 1)));  // at most 17
                __hip_atomic_fetch_add(at + (d >> 2) * S, 1u << (8 * (d & 3)), __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_WORKGROUP);
            }
        }
    }
    __syncthreads();
    low_level<2>(buf1, buf2, run_parities<2>(sr, A), run_parities<2>(sc, A));
    __syncthreads();
    low_level<1>(buf2, buf1, run_parities<1>(sr, A), run_parities<1>(sc, A));
    __syncthreads();
    if (threadIdx.x < run_pairs(0) * run_pairs(0)) {
        constexpr uint32_t RP = run_pairs(0);
        const uint32_t rp = threadIdx.x / RP, cp = threadIdx.x - rp * RP;  // 16 x 16 quads
        uint32_t o[4][6];
        low_quad<0, 6>(buf1, below<0>(sr & 1, 0, rp), below<0>(sc & 1, 0, cp), o);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            uint32_t v[12];
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int x = 0; x < 6; ++x) {
                    const uint32_t a = o[2 * h + s][x / 2], b = o[2 * h + s][3 + x / 2];
                    v[6 * s + x] = x & 1 ? (a >> 16) | (b & 0xFFFF0000u) : (a & 0xFFFFu) | (b << 16);
                }
            uint4 *dst = V + ((uint64_t)(r + 2 * rp + h) * kGrid + c + 2 * cp) / 2 * 3;
#pragma unroll
            for (int x = 0; x < 3; ++x) dst[x] = make_uint4(v[4 * x], v[4 * x + 1], v[4 * x + 2], v[4 * x + 3]);
        }
    }
}

// --- levels 5 .. 4 + F and the histogram ---------------------------------------
constexpr uint32_t kHighThreads = 512;
constexpr int kDwords = 12;       // 24 distances, (w, w + 12) in dword w; 48 bytes a carry pair
constexpr int kQuads = kDwords / 4;
constexpr uint32_t kLowParts = 32 * kTile + 8;  // low parts of a tile's carries, each way, at most

// The twelve dwords of a quad's four outputs, four dwords a round, from nine
// polynomials of 12 dwords.  Times z, dword w - 1 moves to dword w, and
// distance 11 (low half of dword 11) to 12 (high half of dword 0); top: what
// moves from distance 23 to 24.  load(i, x) gives dwords 4i .. 4i + 3 of the
// nine, store(i, o) takes those of the four outputs.
template <class Load, class Store>
__device__ __forceinline__ void high_quad(Load load, Store store, uint32_t (&top)[4]) {
    uint32_t prev[4], last[4][4];
    // dword 11 first: it moves into dword 0
    {
        uint32_t x[3][3][4], y[3][3], zero[4], one[4];
        load(kQuads - 1, x);
#pragma unroll
        for (int w = 0; w < 4; ++w) {
#pragma unroll
            for (int a = 0; a < 3; ++a)
#pragma unroll
                for (int b = 0; b < 3; ++b) y[a][b] = x[a][b][w];
            quad_sums(y, zero, one);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                last[w][q] = w > 0 ? zero[q] + prev[q] : zero[q];
                prev[q] = one[q];
            }
        }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        top[q] = prev[q] >> 16;
        prev[q] <<= 16;
    }
#pragma unroll
    for (int i = 0; i < kQuads - 1; ++i) {
        uint32_t x[3][3][4], y[3][3], zero[4], one[4], o[4][4];
        load(i, x);
#pragma unroll
        for (int w = 0; w < 4; ++w) {
#pragma unroll
            for (int a = 0; a < 3; ++a)
#pragma unroll
                for (int b = 0; b < 3; ++b) y[a][b] = x[a][b][w];
            quad_sums(y, zero, one);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                o[q][w] = zero[q] + prev[q];
                prev[q] = one[q];
            }
        }
        store(i, o);
    }
    uint32_t o[4][4];
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int w = 0; w < 4; ++w) o[q][w] = last[w][q] + (w == 0 ? prev[q] : 0);
    store(kQuads - 1, o);
}

// Output level l from the level below it: src holds 48 bytes a pair, or 24
// bytes (dword x: distances 2x, 2x + 1, 2x + 12, 2x + 13) where BYTES; tops:
// the counters of distance 24, level l = 0 only.
template <int l, bool BYTES>
__device__ __forceinline__ void high_level(const uint32_t *src, uint32_t *dst, uint32_t *tops, uint32_t rpar,
                                           uint32_t cpar) {
    constexpr uint32_t P = run_pairs(l), RP = P << l, D = run_all(l), B = run_all(l + 1);
    for (uint32_t q = threadIdx.x; q < RP * RP; q += kHighThreads) {
        const uint32_t rp = q / RP, cp = q - rp * RP;
        const uint32_t pr = rp / P, tr = rp - pr * P, pc = cp / P, tc = cp - pc * P;
        const Below r = below<l>(rpar, pr, tr), c = below<l>(cpar, pc, tc);
        const uint32_t rows[3] = {r.n * B, r.s0 * B, r.s1 * B}, cols[3] = {c.n, c.s0, c.s1};
        const uint32_t at = (pr * run_len(l) + 2 * tr) * D + pc * run_len(l) + 2 * tc;
        const bool r1 = 2 * tr + 1 < run_len(l), c1 = 2 * tc + 1 < run_len(l);
        uint32_t top[4];
        auto load = [&](int i, uint32_t(&x)[3][3][4]) {
#pragma unroll
            for (int a = 0; a < 3; ++a)
#pragma unroll
                for (int b = 0; b < 3; ++b) {
                    if (BYTES) {
                        const uint2 v = *reinterpret_cast<const uint2 *>(src + (rows[a] + cols[b]) * 6 + 2 * i);
                        x[a][b][0] = v.x & 0x00FF00FFu;
                        x[a][b][1] = (v.x >> 8) & 0x00FF00FFu;
                        x[a][b][2] = v.y & 0x00FF00FFu;
                        x[a][b][3] = (v.y >> 8) & 0x00FF00FFu;
                    } else {
                        const uint4 v = *reinterpret_cast<const uint4 *>(src + (rows[a] + cols[b]) * kDwords + 4 * i);
                        x[a][b][0] = v.x;
                        x[a][b][1] = v.y;
                        x[a][b][2] = v.z;
                        x[a][b][3] = v.w;
                    }
                }
        };
        auto store = [&](int i, const uint32_t(&o)[4][4]) {
            uint32_t *d = dst + at * kDwords + 4 * i;
            *reinterpret_cast<uint4 *>(d) = make_uint4(o[0][0], o[0][1], o[0][2], o[0][3]);
            if (c1) *reinterpret_cast<uint4 *>(d + kDwords) = make_uint4(o[1][0], o[1][1], o[1][2], o[1][3]);
            if (r1) *reinterpret_cast<uint4 *>(d + D * kDwords) = make_uint4(o[2][0], o[2][1], o[2][2], o[2][3]);
            if (r1 && c1)
                *reinterpret_cast<uint4 *>(d + (D + 1) * kDwords) = make_uint4(o[3][0], o[3][1], o[3][2], o[3][3]);
        };
        high_quad(load, store, top);
        if (l == 0) {
            tops[at] = top[0];
            tops[at + 1] = top[1];
            tops[at + D] = top[2];
            tops[at + D + 1] = top[3];
        }
    }
}

// Clears the histogram; lows[t]: the first low part whose carry is at least
// kTile * t, so the low parts of tile t's carries are [lows[t], lows[t + 1]).
__global__ __launch_bounds__(256) void tiles_setup(unsigned long long *__restrict__ hist, uint32_t entries,
                                                   uint32_t *__restrict__ lows, uint32_t nlows, uint32_t A,
                                                   uint32_t T) {
    const uint32_t t = blockIdx.x * 256 + threadIdx.x;
    if (t < entries) hist[t] = 0;
    if (t < nlows) {
        const uint64_t c = (uint64_t)t * kTile;
        lows[t] = c >= A ? 1u << T : (uint32_t)(((c << T) + A - 1) / A);
    }
}

enum TileSet : uint32_t { kAllTiles = 0, kUpperTiles = 1, kDiagonalTiles = 2 };

// The staging of a tile's part of V in LDS: run_all(F) rows of run_all(F)
// pairs, three 8-byte words a pair.  A thread keeps its column and word, and
// takes every kRowsStep-th row.
template <int F>
struct Stage {
    static constexpr uint32_t D = run_all(F), kRow = 3 * D, kRowsStep = kHighThreads / kRow;
    static constexpr int kSteps = (D + kRowsStep - 1) / kRowsStep;
};

// LDS of tiles_high in dwords: histogram, low parts, run starts, then the
// levels; a: F and 2 levels below, or the tile's own; b: the others.
constexpr uint32_t kHighFixed = kRows * kStride + 2 * kLowParts + 64;
constexpr uint32_t level_dwords(int F, int l) {
    return l == F ? run_all(l) * run_all(l) * 6 : run_all(l) * run_all(l) * kDwords + (l == 0 ? kTile * kTile : 0);
}
// levels F, F - 1, ... 0 alternate between the two buffers, F in the first
constexpr uint32_t buffer_dwords(int F, int first) {
    uint32_t m = 0;
    for (int l = first; l >= 0; l -= 2) m = level_dwords(F, l) > m ? level_dwords(F, l) : m;
    return m;
}

// Tiles of the block (R0, C0), ntr x ntc of them, or of a block on the
// diagonal those above or on its diagonal.  flush: tiles between two flushes
// of the LDS counters; a histogram adds `weight` times the counts.
template <int F>
__global__ __launch_bounds__(kHighThreads) void tiles_high(const uint32_t *__restrict__ V,
                                                           const uint32_t *__restrict__ lows, uint32_t A, uint32_t T,
                                                           uint32_t R0, uint32_t C0, uint32_t ntr, uint32_t ntc,
                                                           uint32_t set, uint32_t flush, uint32_t weight,
                                                           uint32_t nbins, unsigned long long *__restrict__ out) {
    extern __shared__ __align__(16) uint32_t lds[];
    uint32_t *const bufa = lds;                                    // levels F, F - 2, ...
    constexpr uint32_t kA = buffer_dwords(F, F), kB = buffer_dwords(F, F - 1);
    uint32_t *const bufb = bufa + ((kA + 3) & ~3u);                // levels F - 1, F - 3, ...
    uint32_t *const hist = bufb + ((kB + 3) & ~3u);                // [kRows][64]
    uint32_t *const low_r = hist + kRows * kStride;                // low parts: own bits, carry - R at bit 24
    uint32_t *const low_c = low_r + kLowParts;
    uint32_t *const start_r = low_c + kLowParts;                   // grid row of each run's first carry
    uint32_t *const start_c = start_r + 32;
    const uint32_t tid = threadIdx.x;
    for (uint32_t b = tid; b < kRows * kStride; b += kHighThreads) hist[b] = 0;
    uint32_t *const mine = hist + (tid & 63);
    const uint32_t mask = (1u << T) - 1;
    const uint32_t count = set == kAllTiles ? ntr * ntc : set == kUpperTiles ? ntr * (ntr - 1) / 2 : ntr;
    auto tile_of = [&](uint32_t t, uint32_t &R, uint32_t &C) {
        uint32_t tr, tc;
        if (set == kAllTiles) {
            tr = t / ntc;
            tc = t - tr * ntc;
        } else if (set == kDiagonalTiles) {
            tr = tc = t;
        } else {
            uint32_t left = t;  // row tr has ntr - 1 - tr tiles
            tr = 0;
            while (left >= ntr - 1 - tr) left -= ntr - 1 - tr++;
            tc = tr + 1 + left;
        }
        R = R0 + tr * kTile;
        C = C0 + tc * kTile;
    };
    auto flush_hist = [&]() {
        __syncthreads();
        for (uint32_t b = tid; b < nbins; b += kHighThreads) {
            unsigned long long s = 0;
            for (uint32_t l = 0; l < 64; ++l) {
                const uint32_t at = b * kStride + ((l + tid) & 63);
                s += hist[at];
                hist[at] = 0;
            }
            if (s) atomicAdd(hist_copy(out, nbins, kHistCopies) + b, s * weight);
        }
        __syncthreads();
    };
    using St = Stage<F>;
    constexpr uint32_t len = run_len(F), W = kGrid >> F;
    const uint32_t srow = tid / St::kRow, sword = tid - srow * St::kRow, scol = sword / 3;
    const bool stages = srow < St::kRowsStep;
    // grid row of a run's first carry, for the tile at (R, C)
    auto starts = [&](uint32_t R, uint32_t C) {
        if (tid < (1u << F)) start_r[tid] = tid * W + ((R + A * tid) >> F) - ((R0 + A * tid) >> F);
        if (tid >= 64 && tid < 64 + (1u << F)) {
            const uint32_t p = tid - 64;
            start_c[p] = p * W + ((C + A * p) >> F) - ((C0 + A * p) >> F);
        }
    };
    uint2 v[St::kSteps];
    auto fetch = [&]() {
        if (!stages) return;
        const uint32_t pc = scol / len;
        const uint32_t col = start_c[pc] + scol - pc * len;
        const uint2 *base = reinterpret_cast<const uint2 *>(V) + (uint64_t)col * 3 + sword - scol * 3;
#pragma unroll
        for (int s = 0; s < St::kSteps; ++s) {
            const uint32_t e = min((uint32_t)s * St::kRowsStep + srow, St::D - 1);
            const uint32_t pr = e / len;
            v[s] = base[(uint64_t)(start_r[pr] + e - pr * len) * (kGrid * 3)];
        }
    };
    // workgroups b, b + 8, ... run on one XCD: they share a run of consecutive
    // tiles, whose parts of V overlap in that XCD's L2
    const uint32_t xcds = min(gridDim.x, 8u), xcd = blockIdx.x % xcds, lane_of = blockIdx.x / xcds;
    const uint32_t step = (gridDim.x + xcds - 1 - xcd) / xcds;
    const uint32_t end = (uint32_t)((uint64_t)count * (xcd + 1) / xcds);
    const uint32_t t0 = (uint32_t)((uint64_t)count * xcd / xcds) + lane_of;
    uint32_t R = 0, C = 0, i0 = 0, ni = 0, j0 = 0, nj = 0, since = 0;
    auto tile_at = [&](uint32_t t) {
        tile_of(t, R, C);
        i0 = lows[R / kTile];
        ni = lows[R / kTile + 1] - i0;
        j0 = lows[C / kTile];
        nj = lows[C / kTile + 1] - j0;
    };
    if (t0 < end) {
        tile_at(t0);
        starts(R, C);
    }
    __syncthreads();
    if (t0 < end) fetch();
    __syncthreads();  // the run starts are read before the loop writes the next tile's
    for (uint32_t t = t0; t < end; t += step) {
        // level 4 and the low parts of this tile into LDS
        if (stages) {
#pragma unroll
            for (int s = 0; s < St::kSteps; ++s) {
                const uint32_t e = s * St::kRowsStep + srow;
                if (e < St::D) reinterpret_cast<uint2 *>(bufa)[e * St::kRow + sword] = v[s];
            }
        }
        for (uint32_t x = tid; x < ni; x += kHighThreads) {
            const uint64_t w = (uint64_t)A * (i0 + x);
            low_r[x] = ((uint32_t)w & mask) | ((uint32_t)(w >> T) - R) << 24;
        }
        for (uint32_t x = tid; x < nj; x += kHighThreads) {
            const uint64_t w = (uint64_t)A * (j0 + x);
            low_c[x] = ((uint32_t)w & mask) | ((uint32_t)(w >> T) - C) << 24;
        }
        const uint32_t thisR = R, thisC = C, pairs = ni * nj, cols = nj;
        if (t + step < end) {
            tile_at(t + step);
            starts(R, C);
        }
        __syncthreads();
        if (t + step < end) fetch();  // the next tile's level 4, in flight meanwhile
        if constexpr (F >= 4) {
            high_level<3, true>(bufa, bufb, nullptr, run_parities<3>(thisR, A), run_parities<3>(thisC, A));
            __syncthreads();
        }
        if constexpr (F >= 3) {
            uint32_t *const src = F == 3 ? bufa : bufb, *const dst = F == 3 ? bufb : bufa;
            high_level<2, F == 3>(src, dst, nullptr, run_parities<2>(thisR, A), run_parities<2>(thisC, A));
            __syncthreads();
        }
        if constexpr (F >= 2) {
            uint32_t *const src = F == 3 ? bufb : bufa, *const dst = F == 3 ? bufa : bufb;
            high_level<1, F == 2>(src, dst, nullptr, run_parities<1>(thisR, A), run_parities<1>(thisC, A));
            __syncthreads();
        }
        uint32_t *const last = F & 1 ? bufb : bufa, *const tops = last + kTile * kTile * kDwords;
        if constexpr (F >= 1) {
            high_level<0, F == 1>(F & 1 ? bufa : bufb, last, tops, thisR & 1, thisC & 1);
            __syncthreads();
        }
        // every pair (i, j) of low parts: the polynomial of their carries,
        // shifted by the distance of their own bits
        const uint32_t magic = (uint32_t)((0x100000000ull + cols - 1) / max(cols, 1u));  // exact: pairs * cols < 2^32
        for (uint32_t x = tid; x < pairs; x += kHighThreads) {
            const uint32_t i = cols == 1 ? x : __umulhi(x, magic), j = x - i * cols;
            const uint32_t a = low_r[i], b = low_c[j];
            const uint32_t s = (a >> 24) * kTile + (b >> 24);
            uint32_t *h = mine + __popc((a ^ b) & 0xFFFFFFu) * kStride;
            auto add = [&](int d, uint32_t n) {
                __hip_atomic_fetch_add(h + d * kStride, n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            };
            if constexpr (F == 0) {
                const uint2 *q = reinterpret_cast<const uint2 *>(last + s * 6);
#pragma unroll
                for (int g = 0; g < 3; ++g) {
                    const uint2 y = q[g];
                    const uint32_t d[2] = {y.x, y.y};
#pragma unroll
                    for (int w = 0; w < 2; ++w) {
                        const int b0 = 4 * g + 2 * w;  // distances of level 4 reach 20
                        add(b0, d[w] & 0xFF);
                        add(b0 + 1, (d[w] >> 8) & 0xFF);
                        if (b0 + 12 <= 20) add(b0 + 12, (d[w] >> 16) & 0xFF);
                        if (b0 + 13 <= 20) add(b0 + 13, d[w] >> 24);
                    }
                }
            } else {
                const uint4 *q = reinterpret_cast<const uint4 *>(last + s * kDwords);
                const uint32_t top = tops[s];
#pragma unroll
                for (int g = 0; g < kQuads; ++g) {
                    const uint4 y = q[g];
                    const uint32_t d[4] = {y.x, y.y, y.z, y.w};
#pragma unroll
                    for (int w = 0; w < 4; ++w) {
                        add(4 * g + w, d[w] & 0xFFFFu);
                        add(4 * g + w + 12, d[w] >> 16);
                    }
                }
                add(24, top);
            }
        }
        __syncthreads();
        if (++since >= flush) {
            flush_hist();
            since = 0;
        }
    }
    flush_hist();
}

size_t high_lds(int F) {
    const uint32_t a = (buffer_dwords(F, F) + 3) & ~3u;
    const uint32_t b = (buffer_dwords(F, F - 1) + 3) & ~3u;
    return (size_t)(a + b + kHighFixed) * sizeof(uint32_t);
}

const void *high_kernel(int F) {
    switch (F) {
    case 0: return reinterpret_cast<const void *>(&tiles_high<0>);
    case 1: return reinterpret_cast<const void *>(&tiles_high<1>);
    case 2: return reinterpret_cast<const void *>(&tiles_high<2>);
    case 3: return reinterpret_cast<const void *>(&tiles_high<3>);
    default: return reinterpret_cast<const void *>(&tiles_high<4>);
    }
}

}  // namespace

bool carry_tiles_plan(uint64_t A, uint32_t k, CarryTilesPlan *p) {
    if (A == 0 || k > 26) return false;
    while ((A & 1) == 0) A >>= 1;
    if (A < 3 || A >= 65536) return false;
    p->A = (uint32_t)A;
    p->k = k;
    const uint32_t bits = 32 - (uint32_t)__builtin_clz((uint32_t)A);
    if (k < bits + kLow) return false;
    p->F = std::min<uint32_t>(k - bits - kLow, 4);
    p->T = k - kLow - p->F;  // low bits taken by the pairs (i, j): each carry has up to 2^(T - bits) + 1 of them
    if (p->T > bits + 4 || p->T > 18) return false;
    p->hb = 32 - (uint32_t)__builtin_clz((uint32_t)A - 1);
    p->nbins = k + p->hb + 1;
    if (p->nbins > kRows) return false;
    p->table_bytes = (uint64_t)kGrid * kGrid * 24 + kMaxLows * sizeof(uint32_t);
    p->hist_entries = hist_copy_stride(p->nbins) * kHistCopies;
    // measured at A = 58659, k = 20 .. 24: 14 ps a carry pair (half of A^2) for
    // tiles_low, 7.5 ps for each further level, 5 ps a pair of low parts, and
    // 8 us of launches and tails a block
    const double blocks = (p->A + kSide - 1) / kSide, states = 0.5 * p->A * p->A;
    p->seconds = 60e-6 + 4e-6 * blocks * (blocks + 1) + (14e-12 + 7.5e-12 * p->F) * states +
                 5e-12 * std::ldexp(1.0, 2 * (int)p->T - 1);
    return true;
}

cr_status carry_tiles_run(const CarryTilesPlan &p, void *table, unsigned long long *hist, int cus,
                          hipStream_t stream) {
    uint32_t *const lows = reinterpret_cast<uint32_t *>(static_cast<char *>(table) + (uint64_t)kGrid * kGrid * 24);
    const uint32_t nlows = p.A / kTile + 2;
    hipLaunchKernelGGL(tiles_setup, dim3(((uint32_t)std::max<uint64_t>(p.hist_entries, nlows) + 255) / 256), dim3(256),
                       0, stream, hist, (uint32_t)p.hist_entries, lows, nlows, p.A, p.T);
    CR_HIP(hipGetLastError());
    const void *k = high_kernel((int)p.F);
    const size_t lds = high_lds((int)p.F);
    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k, (int)kHighThreads, lds) != hipSuccess || per_cu <= 0)
        return fail(CR_ERR_DEVICE, "occupancy query failed for the carry tile kernel");
    // a lane's counter takes a 64th of a tile's pairs of low parts (rounded up
    // to 8 per 512 pairs), each at most 4^8 - 1 (weights apply at the flush)
    const uint64_t m = kTile * (((1ull << p.T) / p.A) + 1);  // low parts of a tile, each way
    if (m > kLowParts) return fail(CR_ERR_DEVICE, "carry tiles: %llu low parts", (unsigned long long)m);
    const uint32_t flush = (uint32_t)std::max<uint64_t>(1, (1ull << 32) / (8 * (m * m / 512 + 1) * 65536) - 1);
    const uint32_t W = kGrid >> p.F;
    for (uint32_t R0 = 0; R0 < p.A; R0 += kSide)
        for (uint32_t C0 = R0; C0 < p.A; C0 += kSide) {
            const uint32_t nr = std::min(kSide, p.A - R0), nc = std::min(kSide, p.A - C0);
            const uint32_t ntr = (nr + kTile - 1) / kTile, ntc = (nc + kTile - 1) / kTile;
            const uint32_t ur = std::min(W, ((ntr * kTile) >> p.F) + 1), uc = std::min(W, ((ntc * kTile) >> p.F) + 1);
            hipLaunchKernelGGL(tiles_low, dim3(kGrid / kTile, kGrid / kTile), dim3(kLowThreads), 0, stream,
                               (uint4 *)table, p.A, R0, C0, p.F, ur, uc);
            CR_HIP(hipGetLastError());
            for (uint32_t s = R0 == C0 ? (uint32_t)kUpperTiles : (uint32_t)kAllTiles;
                 s <= (R0 == C0 ? (uint32_t)kDiagonalTiles : (uint32_t)kAllTiles); ++s) {
                const uint32_t count = s == kAllTiles ? ntr * ntc : s == kUpperTiles ? ntr * (ntr - 1) / 2 : ntr;
                if (count == 0) continue;
                const uint32_t blocks = std::min<uint32_t>(count, (uint32_t)per_cu * (uint32_t)cus);
                const uint32_t *a_V = (const uint32_t *)table, *a_lows = lows;
                uint32_t a_A = p.A, a_T = p.T, a_R0 = R0, a_C0 = C0, a_ntr = ntr, a_ntc = ntc, a_s = s, a_flush = flush,
                         a_w = s == kDiagonalTiles ? 1 : 2, a_nb = p.nbins;
                void *args[] = {(void *)&a_V, (void *)&a_lows, &a_A, &a_T, &a_R0, &a_C0, &a_ntr, &a_ntc, &a_s, &a_flush, &a_w, &a_nb,
                                &hist};
                CR_HIP(hipLaunchKernel(k, dim3(blocks), dim3(kHighThreads), args, lds, stream));
            }
        }
    return CR_OK;
}

}  // namespace cr
