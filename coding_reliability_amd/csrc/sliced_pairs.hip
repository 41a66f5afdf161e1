// Pair-distance histograms of whole codes, 2^k words, 32 pairs an instruction
// (gfx950): the same raw[] as the pair kernel (an_pairs.hip).
//
// For odd A the low k bits lo = A*i mod 2^k run over every residue once, so a
// code is the function h(lo) of the other n - k bits, and a pair (lo, lo ^ x)
// differs in popcount(x) + popcount(h(lo) ^ h(lo ^ x)) places: the k low bits
// cost nothing when x is the same for many pairs.  32 consecutive lo form a
// "word": plane b of a word holds bit b of its 32 h's.  For two words w, v and x
// = (w ^ v, xb), the 32 pairs' distances come from the planes of w and the
// planes of v with their bits permuted by xb: n - k XORs, carry-save adders
// (three-input v_bitop3) down to the bits q0 .. q4 of 32 sums, and a histogram of
// the sums as the counts of the products of q0 .. q3 (v_bcnt accumulates them),
// from which the counts of the values 0 .. 15 follow by inclusion-exclusion.
// 68 instructions for 32 pairs of 16-bit h's, 58 for 15 bits, 54 for 12, 24 for
// 7, where the pair kernel takes 3 and an LDS increment (which bounds it) for
// one.  Bound by VALU issue: 20.3e12 pairs/s for 16-bit multipliers at k = 18
// (9.4e12 in the pair kernel), 43e12 lane instructions/s, where bit counts
// issue at 37e12 and XORs and bitop3 at up to 55e12 (51e12 in this mix); 1024
// mixed codes of 8 to 18 bits 197 ms (473 ms).  A single code of 2^16 words takes
// 0.155 ms (0.34 ms), of 2^14 34 us (64 us); below that four workgroups per
// block of 64 x 64 words are too few, and the short kernel takes over.
//
// The first adders work on triples of planes (p1, p2, p3) stored as p1, p1 ^
// p2, p1 ^ p3, p1 ^ p2 ^ p3, for either side: the sum is one XOR and the
// majority a ^ ((a ^ b) & (a ^ c)) three operations, not five with the XORs.
//
// A workgroup of four waves takes 64 x 64 words (2^22 pairs).  Lane l of a wave
// holds word l of one side permuted by two xb (two sets of registers) and reads
// word l ^ delta of the other from LDS for each delta < 64, in order of
// popcount(delta), so that popcount(x) is the same for the wave and the product
// counts are kept in registers over a popcount class; they are added to LDS
// counters by class (popcount of delta and xb).  The four waves and up to four
// workgroups share the 32 xb, and in small launches up to four the delta.
#include <algorithm>
#include <atomic>

#include "cr_device.h"
#include "cr_internal.h"

namespace cr {
namespace {

using namespace dev;

constexpr uint32_t kThreads = 256;
constexpr int kRecord = 6;        // 16-byte chunks of a word's record: five triples, one plane
constexpr int kProducts = 16;     // product sums of a class: index = set of q0 .. q3; index 0: q4
constexpr uint32_t kClasses = 12; // popcount(delta) + popcount(xb): 0 .. 11
constexpr uint32_t kCols = 32;    // columns of the LDS counters
constexpr uint32_t kHist = 64;

#define CR_XOR3(a, b, c) __builtin_amdgcn_bitop3_b32(a, b, c, 0x96)
#define CR_MAJ3(a, b, c) __builtin_amdgcn_bitop3_b32(a, b, c, 0xE8)

__device__ __forceinline__ void full_add(uint32_t a, uint32_t b, uint32_t c, uint32_t &s, uint32_t &k) {
    s = CR_XOR3(a, b, c);
    k = CR_MAJ3(a, b, c);
}
__device__ __forceinline__ void half_add(uint32_t a, uint32_t b, uint32_t &s, uint32_t &k) {
    s = a ^ b;
    k = a & b;
}

// A word's planes: NP = 16, 15, 12 or 7 of them, NT triples and perhaps one more.
template <int NP>
struct Planes {
    static constexpr int NT = NP / 3;
    static constexpr bool one = NP % 3 == 1;
    uint32_t p[NT], p12[NT], p13[NT], p123[NT], t;
};

// Bits of the 32 sums popcount(planes of a ^ planes of b).
template <int NP>
__device__ __forceinline__ void distances(const Planes<NP> &a, const Planes<NP> &b, uint32_t (&q)[5]) {
    constexpr int NT = Planes<NP>::NT;
    uint32_t s[NT], m[NT];
#pragma unroll
    for (int i = 0; i < NT; ++i) {
        s[i] = a.p123[i] ^ b.p123[i];
        const uint32_t x = a.p12[i] ^ b.p12[i];
        const uint32_t y = __builtin_amdgcn_bitop3_b32(x, a.p13[i], b.p13[i], 0x60);  // x & (a ^ b)
        m[i] = CR_XOR3(y, a.p[i], b.p[i]);
    }
    q[4] = 0;
    if constexpr (NP == 16) {
        uint32_t c0, c1, c2, d, e0, e1, e2, e3, f, g, i0, i1, u, v;
        full_add(s[0], s[1], s[2], u, c0);
        full_add(s[3], s[4], a.t ^ b.t, v, c1);
        half_add(u, v, q[0], c2);
        full_add(m[0], m[1], m[2], d, e0);
        full_add(m[3], m[4], c0, f, e1);
        full_add(c1, c2, d, g, e2);
        half_add(g, f, q[1], e3);
        full_add(e0, e1, e2, u, i0);
        half_add(u, e3, q[2], i1);
        half_add(i0, i1, q[3], q[4]);
    } else if constexpr (NP == 15) {
        uint32_t c0, c1, d, e0, e1, e2, f, u;
        full_add(s[0], s[1], s[2], u, c0);
        full_add(u, s[3], s[4], q[0], c1);
        full_add(m[0], m[1], m[2], d, e0);
        full_add(m[3], m[4], c0, f, e1);
        full_add(d, f, c1, q[1], e2);
        full_add(e0, e1, e2, q[2], q[3]);
    } else if constexpr (NP == 12) {
        uint32_t c0, c1, d, e0, e1, e2, f, u;
        full_add(s[0], s[1], s[2], u, c0);
        half_add(u, s[3], q[0], c1);
        full_add(m[0], m[1], m[2], d, e0);
        full_add(m[3], c0, c1, f, e1);
        half_add(d, f, q[1], e2);
        full_add(e0, e1, e2, q[2], q[3]);
    } else {
        uint32_t c0;
        full_add(s[0], s[1], a.t ^ b.t, q[0], c0);
        full_add(m[0], m[1], c0, q[1], q[2]);
        q[3] = 0;
    }
}

// Adds the counts of the products of q0 .. q3 (bit i of the index: q_i) and of q4.
template <int NP>
__device__ __forceinline__ void count_products(const uint32_t (&q)[5], uint32_t (&acc)[kProducts]) {
    constexpr int B = NP == 7 ? 3 : 4;
    uint32_t prod[1 << B];
#pragma unroll
    for (int x = 1; x < (1 << B); ++x) {
        const int low = x & -x, rest = x ^ low;
        const int bit = __builtin_ctz((unsigned)low);
        prod[x] = rest ? prod[rest] & q[bit] : q[bit];
        acc[x] += __popc(prod[x]);
    }
    if (NP == 16) acc[0] += __popc(q[4]);
}

// Bits of a plane whose positions differ in bit B trade places.
template <int B>
__device__ __forceinline__ uint32_t swap_bits(uint32_t x) {
    if constexpr (B == 4) return __builtin_amdgcn_alignbit(x, x, 16);
    if constexpr (B == 3) return __builtin_amdgcn_perm(x, x, 0x02030001u);
    constexpr uint32_t m = B == 2 ? 0x0F0F0F0Fu : B == 1 ? 0x33333333u : 0x55555555u;
    return ((x >> (1 << B)) & m) | ((x & m) << (1 << B));
}
template <int B, int NP>
__device__ __forceinline__ void swap_planes(Planes<NP> &a) {
#pragma unroll
    for (int i = 0; i < Planes<NP>::NT; ++i) {
        a.p[i] = swap_bits<B>(a.p[i]);
        a.p12[i] = swap_bits<B>(a.p12[i]);
        a.p13[i] = swap_bits<B>(a.p13[i]);
        a.p123[i] = swap_bits<B>(a.p123[i]);
    }
    if (Planes<NP>::one) a.t = swap_bits<B>(a.t);
}

struct Lds {
    uint32_t rec[kRecord * 64 * 4];                          // records of the row words, [chunk][word][4]
    uint32_t plane[16 * 64];                                 // planes of 64 words being generated
    uint32_t count[kClasses * kProducts * kCols];
    uint32_t sum[kClasses * kProducts];
    uint32_t pairs[kClasses];
    unsigned long long hist[kHist];
    unsigned long long item;
};

// Bit i of byte j of the eight bytes of x (lower four) and y trades places with
// bit j of byte i.
__device__ __forceinline__ void transpose8(uint32_t &x, uint32_t &y) {
    auto step = [](uint32_t &v, uint32_t shift, uint32_t mask) {
        const uint32_t t = (v ^ (v >> shift)) & mask;
        v = CR_XOR3(v, t, t << shift);
    };
    step(x, 7, 0x00AA00AAu);
    step(y, 7, 0x00AA00AAu);
    step(x, 14, 0x0000CCCCu);
    step(y, 14, 0x0000CCCCu);
    const uint32_t t = (x ^ (y << 4)) & 0xF0F0F0F0u;
    x ^= t;
    y ^= t >> 4;
}

// The planes of words 64 * block + l: thread (l, q) takes elements 8q .. 8q + 7
// of its word, h advanced as in the spectral generator (see next_high there).
__device__ __forceinline__ void generate(Lds &L, const SlicedJob &job, uint32_t block) {
    const uint32_t l = threadIdx.x & 63, q = threadIdx.x >> 6;
    const uint32_t lo = ((block * 64 + l) << 5) + 8 * q;
    const uint32_t i = (lo * job.Ainv) & ((1u << job.k) - 1);
    uint32_t h = (uint32_t)(((uint64_t)job.A * i) >> job.k);
    uint32_t two[4];  // elements 2e, 2e + 1
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        two[e / 2] = e & 1 ? two[e / 2] | h << 16 : h;
        const uint32_t t = h + job.tc;
        h = min(t, t - job.A);
    }
    // bytes of the planes 0 .. 7 and 8 .. 15
    uint32_t low[2], high[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        low[e] = __builtin_amdgcn_perm(two[2 * e + 1], two[2 * e], 0x06040200u);
        high[e] = __builtin_amdgcn_perm(two[2 * e + 1], two[2 * e], 0x07050301u);
    }
    transpose8(low[0], low[1]);
    transpose8(high[0], high[1]);
    uint8_t *const at = reinterpret_cast<uint8_t *>(L.plane) + l * 4 + q;
#pragma unroll
    for (int b = 0; b < 8; ++b) {
        at[b * 256] = (uint8_t)(low[b / 4] >> (8 * (b & 3)));
        at[(b + 8) * 256] = (uint8_t)(high[b / 4] >> (8 * (b & 3)));
    }
}

template <int NP>
__device__ __forceinline__ void load_planes(const Lds &L, Planes<NP> &a) {
    const uint32_t l = threadIdx.x & 63;
#pragma unroll
    for (int i = 0; i < Planes<NP>::NT; ++i) {
        const uint32_t p1 = L.plane[(3 * i) * 64 + l], p2 = L.plane[(3 * i + 1) * 64 + l],
                       p3 = L.plane[(3 * i + 2) * 64 + l];
        a.p[i] = p1;
        a.p12[i] = p1 ^ p2;
        a.p13[i] = p1 ^ p3;
        a.p123[i] = p1 ^ p2 ^ p3;
    }
    a.t = Planes<NP>::one ? L.plane[(NP - 1) * 64 + l] : 0;
}

// One item: words of block `col` in registers against those of block `row`.
template <int NP>
__device__ void run_item(Lds &L, const SlicedJob &job, uint32_t row, uint32_t col, uint32_t part) {
    const uint32_t l = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    generate(L, job, col);
    __syncthreads();
    Planes<NP> a, b;
    load_planes<NP>(L, a);
    __syncthreads();
    if (row != col) {
        generate(L, job, row);
        __syncthreads();
    }
    {
        Planes<NP> r;
        load_planes<NP>(L, r);
#pragma unroll
        for (int c = 0; c < Planes<NP>::NT; ++c)
            if ((uint32_t)(c & 3) == wave)
                reinterpret_cast<uint4 *>(L.rec)[c * 64 + l] = make_uint4(r.p[c], r.p12[c], r.p13[c], r.p123[c]);
        if (wave == 3) L.rec[(kRecord - 1) * 256 + l] = r.t;
    }
    // the xb of this wave: index bits 0 .. 3 are bits 3, 4, 2, 1 of xb, so that
    // the steps of a Gray code are one byte or half-word move; each with xb's
    // bit 0 off (a) and on (b)
    const uint32_t xparts = min(job.parts, 4u), per = 4 / xparts, first = (part % xparts * 4 + wave) * per;
    // and of the 64 delta those whose upper bits are the rest of the part
    const uint32_t dbits = job.parts == 16 ? 4 : job.parts == 8 ? 5 : 6, dhigh = (part / xparts) << dbits;
    const uint32_t base = __popc(dhigh);
    if (first & 1) swap_planes<3>(a);
    if (first & 2) swap_planes<4>(a);
    if (first & 4) swap_planes<2>(a);
    if (first & 8) swap_planes<1>(a);
    b = a;
    swap_planes<0>(b);
    __syncthreads();
    for (uint32_t j = 0; j < per; ++j) {
        const uint32_t index = first ^ (j ^ (j >> 1));
        const uint32_t xbits = __popc(index);
        uint32_t delta = 0;
        for (uint32_t pd = 0; pd <= dbits; ++pd) {
            uint32_t acca[kProducts] = {}, accb[kProducts] = {};
            const uint32_t last = ((1u << dbits) - 1) & ~((1u << (dbits - pd)) - 1);  // the largest with pd bits
            delta = (1u << pd) - 1;
            uint32_t n = 0;
            for (;;) {
                const uint32_t from = l ^ (delta | dhigh);
                const uint4 *rec = reinterpret_cast<const uint4 *>(L.rec) + from;
                Planes<NP> r;
#pragma unroll
                for (int c = 0; c < Planes<NP>::NT; ++c) {
                    const uint4 y = rec[c * 64];
                    r.p[c] = y.x;
                    r.p12[c] = y.y;
                    r.p13[c] = y.z;
                    r.p123[c] = y.w;
                }
                r.t = Planes<NP>::one ? L.rec[(kRecord - 1) * 256 + from] : 0;
                uint32_t q[5];
                distances<NP>(a, r, q);
                count_products<NP>(q, acca);
                distances<NP>(b, r, q);
                count_products<NP>(q, accb);
                ++n;
                if (delta == last) break;
                // the next larger number with as many bits
                const uint32_t c = delta & (0u - delta), up = delta + c;
                delta = up | (((up ^ delta) >> 2) >> __builtin_ctz(c));
            }
            uint32_t *at = L.count + (base + pd + xbits) * (kProducts * kCols) + (l & (kCols - 1));
#pragma unroll
            for (int x = 0; x < kProducts; ++x) {
                if (x == 0 ? NP != 16 : NP == 7 && x >= 8) continue;
                __hip_atomic_fetch_add(at + x * kCols, acca[x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                __hip_atomic_fetch_add(at + (kProducts + x) * kCols, accb[x], __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_WORKGROUP);
            }
            if (l == 0) {
                __hip_atomic_fetch_add(L.pairs + base + pd + xbits, n * 2048, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                __hip_atomic_fetch_add(L.pairs + base + pd + xbits + 1, n * 2048, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_WORKGROUP);
            }
        }
        const uint32_t flip = ((j + 1) & 1) ? 3 : 4;  // per <= 4: index bits 0 and 1
        if (j + 1 < per) {
            if (flip == 3) {
                swap_planes<3>(a);
                swap_planes<3>(b);
            } else {
                swap_planes<4>(a);
                swap_planes<4>(b);
            }
        }
    }
}

// Class sums into the workgroup's histogram.  A block against itself has
// every unordered pair twice (and each element with itself, distance 0).
__device__ void finish_item(Lds &L, uint32_t base, bool twice) {
    __syncthreads();
    if (threadIdx.x < kClasses * kProducts) {
        uint32_t s = 0;
#pragma unroll 8
        for (uint32_t c = 0; c < kCols; ++c) {
            const uint32_t at = threadIdx.x * kCols + ((c + threadIdx.x) & (kCols - 1));
            s += L.count[at];
            L.count[at] = 0;
        }
        L.sum[threadIdx.x] = s;
    }
    __syncthreads();
    if (threadIdx.x < kClasses) {
        const uint32_t cls = threadIdx.x;
        uint32_t v[kProducts];
        const uint32_t sixteen = L.sum[cls * kProducts];
#pragma unroll
        for (int x = 1; x < kProducts; ++x) v[x] = L.sum[cls * kProducts + x];
        v[0] = L.pairs[cls];
        L.pairs[cls] = 0;
#pragma unroll
        for (int b = 1; b < kProducts; b <<= 1)
#pragma unroll
            for (int x = 0; x < kProducts; ++x)
                if (!(x & b)) v[x] -= v[x | b];
        v[0] -= sixteen;
        const uint32_t shift = twice ? 1 : 0;
        auto add = [&](uint32_t d, uint32_t n) {
            if (n && d) atomicAdd(&L.hist[d], (unsigned long long)(n >> shift));
        };
#pragma unroll
        for (int x = 0; x < kProducts; ++x) add(base + cls + x, v[x]);
        add(base + cls + 16, sixteen);
    }
    __syncthreads();
}

// jobs: device array, or null for the one job `single`, whose histogram goes
// to `direct`.
__global__ __launch_bounds__(kThreads) void sliced_kernel(const SlicedJob *__restrict__ jobs, uint32_t njobs,
                                                          uint64_t total_items,
                                                          unsigned long long *__restrict__ counter,
                                                          const SlicedJob single, const DirectResult direct) {
    __shared__ Lds L;
    if (!jobs) direct_start(direct);
    const uint32_t tid = threadIdx.x;
    for (uint32_t i = tid; i < kClasses * kProducts * kCols; i += kThreads) L.count[i] = 0;
    if (tid < kClasses) L.pairs[tid] = 0;
    if (tid < kHist) L.hist[tid] = 0;
    __syncthreads();
    uint32_t cur = 0xFFFFFFFFu;
    auto flush = [&]() {
        if (cur == 0xFFFFFFFFu) return;
        const SlicedJob &job = jobs ? jobs[cur] : single;
        if (tid < job.nbins && tid < kHist) {
            const unsigned long long n = L.hist[tid];
            if (n) atomicAdd(hist_copy(job.out, job.nbins, job.out_copies) + tid, n);
            L.hist[tid] = 0;
        }
        __syncthreads();
    };
    for (uint64_t t = blockIdx.x; t < total_items;) {
        uint32_t jb = jobs ? cur : 0;
        if (jobs && (cur == 0xFFFFFFFFu || t < jobs[cur].item_begin || t >= jobs[cur].item_begin + jobs[cur].items)) {
            uint32_t lo = 0, hi = njobs - 1;
            while (lo < hi) {
                const uint32_t mid = (lo + hi + 1) >> 1;
                if (jobs[mid].item_begin <= t) lo = mid; else hi = mid - 1;
            }
            jb = uniform32(lo);
        }
        if (jb != cur) {
            flush();
            cur = jb;
        }
        const SlicedJob &job = jobs ? jobs[jb] : single;
        const uint32_t local = uniform32((uint32_t)(t - job.item_begin));
        const uint32_t part = local % job.parts, pair = local / job.parts;
        // pair = col (col + 1) / 2 + row, row <= col
        uint32_t col = (uint32_t)((sqrtf(8.0f * (float)pair + 1.0f) - 1.0f) * 0.5f);
        while (col * (col + 1) / 2 > pair) --col;
        while ((col + 1) * (col + 2) / 2 <= pair) ++col;
        col = uniform32(col);
        const uint32_t row = pair - col * (col + 1) / 2;
        if (job.planes > 15)
            run_item<16>(L, job, row, col, part);
        else if (job.planes > 12)
            run_item<15>(L, job, row, col, part);
        else if (job.planes > 7)
            run_item<12>(L, job, row, col, part);
        else
            run_item<7>(L, job, row, col, part);
        finish_item(L, __popc(row ^ col), row == col);
        if (tid == 0) L.item = counter ? (unsigned long long)gridDim.x + atomicAdd(counter, 1ull) : t + gridDim.x;
        __syncthreads();
        t = uniform64(L.item);
        __syncthreads();
    }
    flush();
    if (!jobs) direct_finish(direct, single.nbins, L.sum);
}

}  // namespace

bool sliced_job(uint64_t A, uint64_t num_words, SlicedJob *j) {
    if (A == 0 || num_words < 2048 || (num_words & (num_words - 1)) || num_words > (1ull << 24)) return false;
    while ((A & 1) == 0) A >>= 1;
    if (A >> 17) return false;
    const uint32_t k = (uint32_t)__builtin_ctzll(num_words);
    const uint64_t top = A * (num_words - 1);
    uint32_t n = 64 - (uint32_t)__builtin_clzll(top);
    if (n < k) n = k;
    if (n - k > 16) return false;
    uint32_t x = (uint32_t)A;
    for (int i = 0; i < 5; ++i) x *= 2u - (uint32_t)A * x;  // inverse modulo 2^32
    *j = SlicedJob{};
    j->A = (uint32_t)A;
    j->Ainv = x & (uint32_t)(num_words - 1);
    j->tc = (uint32_t)((A * j->Ainv - 1) >> k);
    j->k = k;
    j->planes = n - k;
    j->parts = 1;
    return true;
}

// A = 58659, 32767, 8191 and 127 at k = 16 .. 19.
double sliced_rate(const SlicedJob &j) {
    return j.planes > 15 ? 19e12 : j.planes > 12 ? 23e12 : j.planes > 7 ? 25e12 : 45e12;
}

// Resident workgroups per CU (one query per process: the answer is a property
// of the kernel and of gfx950's CU).
static uint32_t sliced_per_cu() {
    static std::atomic<int> cache{0};
    int n = cache.load(std::memory_order_relaxed);
    if (n > 0) return (uint32_t)n;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, reinterpret_cast<const void *>(&sliced_kernel), (int)kThreads,
                                                     0) != hipSuccess ||
        n <= 0)
        return 0;
    cache.store(n, std::memory_order_relaxed);
    return (uint32_t)n;
}

void sliced_ranges(std::vector<SlicedJob> &jobs, int cus, uint64_t *total_items) {
    auto blocks = [](const SlicedJob &j) {
        const uint64_t b = 1ull << (j.k - 11);
        return b * (b + 1) / 2;
    };
    uint64_t whole = 0;
    for (const SlicedJob &j : jobs) whole += blocks(j);
    // an item of a whole block keeps a workgroup busy for some 0.2 ms on a full
    // CU: below 8 per resident workgroup the blocks are split in four by xb
    // (which generates the words four times, 4 % more), and the smallest
    // launches further by delta: 2^15 words 67 us with 4 or 16 parts and 61 with
    // 8, 2^14 42 us with 4 and 34 with 16; 2^16 166 us with 8, 157 with 4
    const uint64_t resident = (uint64_t)std::max(sliced_per_cu(), 1u) * (uint64_t)cus;
    const uint32_t parts = whole * 16 < resident ? 16 : whole * 4 < resident ? 8 : whole < 8 * resident ? 4 : 1;
    uint64_t at = 0;
    for (SlicedJob &j : jobs) {
        j.parts = parts;
        j.items = blocks(j) * parts;
        j.item_begin = at;
        at += j.items;
    }
    *total_items = at;
}

cr_status launch_sliced(const SlicedJob *d_jobs, uint32_t njobs, uint64_t total_items, unsigned long long *counter,
                        int cus, hipStream_t stream) {
    if (njobs == 0 || total_items == 0) return CR_OK;
    const uint32_t per_cu = sliced_per_cu();
    if (per_cu == 0) return fail(CR_ERR_DEVICE, "occupancy query failed for the sliced pair kernel");
    const uint32_t blocks = (uint32_t)std::min<uint64_t>(total_items, (uint64_t)per_cu * (uint32_t)cus);
    hipLaunchKernelGGL(sliced_kernel, dim3(blocks), dim3(kThreads), 0, stream, d_jobs, njobs, total_items, counter,
                       SlicedJob{}, DirectResult{});
    CR_HIP(hipGetLastError());
    return CR_OK;
}

cr_status launch_sliced_direct(const SlicedJob &job, uint64_t items, const dev::DirectResult &out, int cus,
                               hipStream_t stream) {
    const uint32_t per_cu = sliced_per_cu();
    if (per_cu == 0) return fail(CR_ERR_DEVICE, "occupancy query failed for the sliced pair kernel");
    const uint32_t blocks = (uint32_t)std::min<uint64_t>(items, (uint64_t)per_cu * (uint32_t)cus);
    hipLaunchKernelGGL(sliced_kernel, dim3(blocks), dim3(kThreads), 0, stream, (const SlicedJob *)nullptr, 1u, items,
                       out.queue, job, out);
    CR_HIP(hipGetLastError());
    return CR_OK;
}

}  // namespace cr
