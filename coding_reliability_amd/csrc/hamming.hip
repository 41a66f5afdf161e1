// Extended-Hamming weight histograms and AN Monte Carlo pair histograms (gfx950).
//
// Hamming: by linearity the distance distribution of the code is the weight
// distribution of its codewords (the reference's method,
// distance_distribution/src/hamming.cu:183-208), so the kernel histograms the
// weight of the non-extended codeword, popcount(d) + sum_t parity(d & mask_t)
// (computeHamming<N>, hamming.cu:39-59), over a stream of data words d:
//   stride  d = (first + s*stride) mod 2^k      (integer grid)
//   list    d = list[s]                         (the reference grid's sample points)
//   mc      d = Philox word s of (seed, stream) (replaces dhamming_mc's cuRAND draw)
// (Ranges of consecutive words, dhamming's exhaustive mode, hamming.cu:64-81, need
// no enumeration, see hamming_range.hip; a few words come here as a grid of stride 1.)
// AN Monte Carlo: every word A*i against m Philox samples A*u_ij
// (replaces dancoding_mc_shared, an_coding_mc.cu:94-158).
#include <algorithm>
#include <atomic>
#include <type_traits>

#include "cr_device.h"
#include "cr_internal.h"

namespace cr {
namespace {

using namespace dev;

// Work item = 64 lanes x job.lane_samples samples.  Items of up to 2^18 words
// keep the work-queue counter (one device-scope atomic per item) below its
// throughput limit (about 8e7 items/s); small jobs use smaller items so that
// they still fill the device.

// Syndrome tables: the syndrome (bit t = parity(d & m_t)) is linear over
// GF(2), so it is the XOR of the syndromes of the data word's bytes; table f
// holds the syndromes of byte f's 256 values, one byte each: 4 tables for 32-bit
// data, 8 for 64-bit.  A 256-byte table has two dwords in every LDS bank, so
// most lookups take two passes (the LDS is then busy nearly as long as the
// VALU), where five 7-bit fields a half word would take one; but those need
// more instructions and registers.  (39,32) Monte Carlo of 2^34 words with
// fields of 8 / 7 / 6 bits: 9.0 / 9.8 / 11.2 ms, (72,64) of 2^30 1.24 / 1.39 /
// 1.47 ms, a (39,32) stride grid of 2^30 0.43 / 0.46 / 0.47 ms.  With 7 bits,
// two-operand XORs and scalar Philox keys: 10.6, 1.40 and 0.50 ms.
constexpr uint32_t kBits = 8, kFields = 4;  // of a field; fields per 32-bit half
constexpr uint32_t kTable = 1u << kBits;

template <bool W64>
constexpr uint32_t kTabBytes = (W64 ? 2 : 1) * kFields * kTable;

template <bool W64>
__device__ void build_tables(uint8_t *tab, const uint64_t *masks) {
    uint64_t m[7];
#pragma unroll
    for (int t = 0; t < 7; ++t) m[t] = masks[t];
    for (uint32_t e = threadIdx.x; e < kTabBytes<W64>; e += 64) {
        const uint32_t f = e / kTable;
        const uint64_t x = (uint64_t)(e % kTable) << (32 * (f / kFields) + kBits * (f % kFields));
        uint32_t syn = 0;
#pragma unroll
        for (int t = 0; t < 7; ++t) syn |= (uint32_t)(__popcll(x & m[t]) & 1) << t;
        tab[e] = (uint8_t)syn;
    }
    __syncthreads();
}

// The table lookups of U words (all issued before any is combined, so they
// are in flight together) and their combination into weights: popcount of the
// data word plus popcount of the syndrome, the weight of the non-extended
// codeword.
template <bool W64, int U>
__device__ __forceinline__ void table_reads(const uint64_t (&d)[U], const uint8_t *tab,
                                            uint32_t (&r)[U][(W64 ? 2 : 1) * kFields]) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
        for (uint32_t f = 0; f < (W64 ? 2 : 1) * kFields; ++f) {
            const uint32_t x = (uint32_t)(d[u] >> (32 * (f / kFields)));
            r[u][f] = tab[kTable * f + ((x >> (kBits * (f % kFields))) & (kTable - 1))];
        }
}

// FULL: dmask covers the whole word (k = 32 or 64), so the AND is left out.
template <bool W64, int U, bool FULL = false>
__device__ __forceinline__ void table_weights(const uint64_t (&d)[U], uint64_t dmask,
                                              const uint32_t (&r)[U][(W64 ? 2 : 1) * kFields], uint32_t (&w)[U]) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
        constexpr uint32_t F = (W64 ? 2 : 1) * kFields;
        uint32_t syn = r[u][0];
#pragma unroll
        for (uint32_t f = 1; f + 1 < F; f += 2) syn = __builtin_amdgcn_bitop3_b32(syn, r[u][f], r[u][f + 1], 0x96);
        if (F % 2 == 0) syn ^= r[u][F - 1];
        const uint64_t dm = FULL ? d[u] : d[u] & dmask;
        w[u] = __popc(syn) + (W64 ? (uint32_t)__popcll(dm) : (uint32_t)__popc((uint32_t)dm));
    }
}

template <bool W64, int U>
__device__ __forceinline__ void weights_tab(const uint64_t (&d)[U], uint64_t dmask, const uint8_t *tab,
                                            uint32_t (&w)[U]) {
    uint32_t r[U][(W64 ? 2 : 1) * kFields];
    table_reads<W64, U>(d, tab, r);
    table_weights<W64, U>(d, dmask, r, w);
}

// One Monte Carlo item: lane l takes the Philox blocks B0 + 64q + l, q <
// spl/PER, B0 = (first + base)/PER (PER = 4 words per block for k <= 32, 2
// for k > 32: sample s of the job is word s mod PER of block s/PER).  Three
// blocks are in flight: at step q the table lookups of block q+1 are issued,
// then the Philox rounds of block q+2 run interleaved with the combination
// of block q, whose lookups were issued a step earlier.  The last two steps
// generate and look up blocks past the item's end, which are not counted.
// CHECK: the item reaches past the job's sample count, so samples >= count
// go to the dummy row.
template <uint32_t PER>
__device__ __forceinline__ void mc_words(const uint32_t (&c)[4], uint64_t (&x)[PER]) {
#pragma unroll
    for (uint32_t u = 0; u < PER; ++u)
        x[u] = PER == 4 ? (uint64_t)c[u] : ((uint64_t)c[2 * u] | ((uint64_t)c[2 * u + 1] << 32));
}

__device__ __forceinline__ void mc_block(uint32_t (&c)[4], uint64_t b, uint32_t stream, const PhiloxKeys &keys) {
    c[0] = (uint32_t)b;
    c[1] = (uint32_t)(b >> 32);
    c[2] = stream;
    c[3] = kMcTag;
    philox_rounds<0>(c, keys);
}

template <bool W64, uint32_t PER, bool CHECK, bool FULL>
__device__ __forceinline__ void mc_blocks(uint32_t *lane_col, const uint8_t *tab, const HamJob &job, uint64_t base,
                                          uint32_t spl, uint64_t count, uint64_t dmask, uint32_t dummy) {
    constexpr uint32_t F = (W64 ? 2 : 1) * kFields;
    const uint32_t lane = threadIdx.x;
    const PhiloxKeys keys = philox_keys(job.seed);
    const uint32_t nq = spl / PER;
    const uint64_t b0 = (job.first + base) / PER + lane;
    uint32_t c[4];
    uint64_t x[2][PER];
    uint32_t r[2][PER][F];
    mc_block(c, b0, job.stream, keys);
    mc_words<PER>(c, x[0]);
    table_reads<W64, PER>(x[0], tab, r[0]);
    mc_block(c, b0 + 64, job.stream, keys);
    // nq is even (spl is a power of two >= 16): two steps per iteration, the
    // buffers of blocks q and q+1 trading places
    for (uint32_t q = 0; q < nq; q += 2) {
#pragma unroll
        for (uint32_t h = 0; h < 2; ++h) {
            mc_words<PER>(c, x[h ^ 1]);
            table_reads<W64, PER>(x[h ^ 1], tab, r[h ^ 1]);
            mc_block(c, b0 + 64ull * (q + h + 2), job.stream, keys);
            uint32_t w[PER];
            table_weights<W64, PER, FULL>(x[h], dmask, r[h], w);
            const uint64_t s = base + ((uint64_t)(q + h) * 64 + lane) * PER;  // first local sample of this lane
#pragma unroll
            for (uint32_t u = 0; u < PER; ++u)
                lds_inc(lane_col + ((!CHECK || s + u < count) ? w[u] : dummy) * kStride);
        }
    }
}

template <bool W64, bool CHECK>
__device__ __forceinline__ void mc_item(uint32_t *lane_col, const uint8_t *tab, const HamJob &job, uint64_t base,
                                        uint32_t spl, uint64_t count, uint64_t dmask, uint32_t dummy) {
    if (!W64 || job.k <= 32) {
        if (job.k == 32)
            mc_blocks<W64, 4, CHECK, true>(lane_col, tab, job, base, spl, count, dmask, dummy);
        else
            mc_blocks<W64, 4, CHECK, false>(lane_col, tab, job, base, spl, count, dmask, dummy);
    } else if (job.k == 64) {
        mc_blocks<W64, 2, CHECK, true>(lane_col, tab, job, base, spl, count, dmask, dummy);
    } else {
        mc_blocks<W64, 2, CHECK, false>(lane_col, tab, job, base, spl, count, dmask, dummy);
    }
}

// Stride and list items.  Lane l takes the words d_q = first + (base + 64q +
// l) * stride for q < spl, so d advances by 64*stride per step (modulo 2^64, or
// 2^32 for k <= 32: only the low k bits reach the weight), or list[base + 64q +
// l].
// kSeqUnroll steps per iteration, all table reads (and list loads) of the
// batch issued before its increments, so the reads overlap instead of each
// waiting behind the previous increment (8 steps of 4 lookups for 32-bit
// words, 4 of 8 for 64-bit).  spl is a multiple of kSeqUnroll.
// CHECK: steps past the job's count go to the dummy row.
template <bool W64>
constexpr uint32_t kSeqUnroll = W64 ? 4 : 8;

template <bool W64, bool CHECK, bool LIST>
__device__ __forceinline__ void seq_item(uint32_t *lane_col, const uint8_t *tab, const HamJob &job, uint64_t base,
                                         uint32_t spl, uint64_t count, uint64_t dmask, uint32_t dummy) {
    using word_t = typename std::conditional<W64, uint64_t, uint32_t>::type;
    const uint32_t lane = threadIdx.x;
    const uint64_t rem = count - base;
    const uint32_t left = rem < 64ull * spl ? (uint32_t)rem : 64u * spl;  // valid samples in the item
    const uint64_t stride = job.stride;
    word_t d = (word_t)(job.first + (base + lane) * stride);
    const word_t step = (word_t)(64 * stride);
    const uint64_t *list = LIST ? job.list + base + lane : nullptr;
    constexpr uint32_t U = kSeqUnroll<W64>;
    for (uint32_t q = 0; q < spl; q += U) {
        uint64_t x[U];
        uint32_t w[U];
        if (LIST) {
#pragma unroll
            for (uint32_t u = 0; u < U; ++u)
                x[u] = (!CHECK || (q + u) * 64 + lane < left) ? list[(q + u) * 64] : 0;
        } else {
#pragma unroll
            for (uint32_t u = 0; u < U; ++u) {
                x[u] = (uint64_t)d;
                d += step;
            }
        }
        weights_tab<W64, U>(x, dmask, tab, w);
#pragma unroll
        for (uint32_t u = 0; u < U; ++u)
            lds_inc(lane_col + ((!CHECK || (q + u) * 64 + lane < left) ? w[u] : dummy) * kStride);
    }
}

__device__ __forceinline__ unsigned long long *copy_out(const HamJob &job) {
    return hist_copy(job.out, job.nbins, job.out_copies);
}

__device__ __forceinline__ uint32_t find_job(const HamJob *jobs, uint32_t njobs, uint64_t t, uint32_t cur) {
    if (cur != 0xFFFFFFFFu && t >= jobs[cur].item_begin && t < jobs[cur].item_begin + jobs[cur].items) return cur;
    uint32_t lo = 0, hi = njobs - 1;
    while (lo < hi) {
        const uint32_t mid = (lo + hi + 1) >> 1;
        if (jobs[mid].item_begin <= t) lo = mid; else hi = mid - 1;
    }
    return uniform32(lo);
}

// ONE: the one job `single`, whose histogram goes to `direct`, in place of the
// device array.
template <bool W64, bool ONE>
__global__ __launch_bounds__(64) void ham_kernel(const HamJob *__restrict__ jobs, uint32_t njobs, uint64_t total_items,
                                                 unsigned long long *__restrict__ counter, uint32_t lds_rows,
                                                 const HamJob single, const DirectResult direct) {
    // the tables at a fixed LDS address (their offsets fold into the reads),
    // the histogram rows in the dynamic LDS after them
    __shared__ uint8_t tab[kTabBytes<W64>];
    extern __shared__ uint32_t lds[];
    const uint32_t lane = threadIdx.x;
    if (ONE) direct_start(direct);
    lds_clear(lds, lds_rows);
    uint32_t *const lane_col = lds + lane;
    const uint32_t dummy = lds_rows - 1;
    uint32_t cur = 0xFFFFFFFFu;
    uint64_t pending = 0;
    auto flush = [&] {
        if (cur == 0xFFFFFFFFu) return;
        const HamJob &job = ONE ? single : jobs[cur];
        flush_rows(lds, 0, job.nbins, copy_out(job));
    };

    for (uint64_t t = first_item(); t < total_items; t = following_item(counter, t)) {
        const uint32_t jb = ONE ? 0 : find_job(jobs, njobs, t, cur);
        const HamJob &job = ONE ? single : jobs[jb];
        const uint32_t spl = job.lane_samples;
        if (jb != cur || pending + spl >= 0xFFFFFFFFull) {
            flush();
            if (jb != cur) build_tables<W64>(tab, job.masks);
            cur = jb;
            pending = 0;
        }
        pending += spl;
        const uint64_t dmask = job.k >= 64 ? ~0ull : ((1ull << job.k) - 1);
        const uint64_t base = (t - job.item_begin + job.item_offset) * (64ull * spl);  // first sample of the item
        const uint64_t count = job.count;

        if (job.source == kHamMc) {
            if (base + 64ull * spl <= count)
                mc_item<W64, false>(lane_col, tab, job, base, spl, count, dmask, dummy);
            else
                mc_item<W64, true>(lane_col, tab, job, base, spl, count, dmask, dummy);
        } else {
            const bool full = base + 64ull * spl <= count;
            if (job.source == kHamList) {
                if (full)
                    seq_item<W64, false, true>(lane_col, tab, job, base, spl, count, dmask, dummy);
                else
                    seq_item<W64, true, true>(lane_col, tab, job, base, spl, count, dmask, dummy);
            } else if (full) {
                seq_item<W64, false, false>(lane_col, tab, job, base, spl, count, dmask, dummy);
            } else {
                seq_item<W64, true, false>(lane_col, tab, job, base, spl, count, dmask, dummy);
            }
        }
    }
    flush();
    if (ONE) direct_finish(direct, single.nbins, lds);
}

// AN Monte Carlo: item = (row block of 64*RM words, sample chunk [j0,
// j0+CJ)).  Row i draws u_ij from the Philox block b of counter
// (b, b >> 32, i mod 2^32, tag ^ (i >> 32)), key (seed, seed >> 32):
//   n <= 32: b = j/4, word j%4, masked to n bits;
//   n >  32: b = j/2, words 2(j%2) (low) and 2(j%2)+1 (high), masked to n bits;
// the codewords A*i and A*u_ij are compared.
constexpr int RM = 4;
constexpr uint32_t kMaxChunk = 256;  // most samples per item (CJ: a power of two, 4 or more)

// One AN Monte Carlo item: samples [jlo, j1) of the chunk that starts at j0
// (a multiple of CJ, so of the words per Philox block: the upper half of the
// block number is the item's).  WIDTH 0: every codeword fits 32 bits (32-bit
// multiply, xor and popcount), 1: the multiplier does, 2: any.  S64: 64-bit
// samples (n > 32).  The first two rounds split into what depends on the row,
// computed once, and what depends on the block number, scalar but for S64.
// Bound by VALU issue: 3.16e12 pairs/s at A = 61 (24-bit samples, long launches; 2.2e12 with whole
// rounds, scalar keys and a 64-bit sample counter), 2.5e12 at A = 58659, n = 24.  CHECK: rows past 2^n and samples outside [jlo, j1) (a partial
// chunk) go to the dummy row; without CHECK, jlo = j0 and j1 - j0 is a
// multiple of the words per Philox block.
template <int WIDTH, bool S64, bool CHECK>
__device__ __forceinline__ void an_mc_item(uint32_t *lane_col, uint64_t A, uint64_t rb, uint64_t nwords, uint64_t j0,
                                           uint64_t jlo, uint64_t j1, uint64_t smask, uint64_t seed,
                                           const PhiloxKeys &keys, uint32_t dummy) {
    constexpr uint32_t M0 = 0xD2511F53u, M1 = 0xCD9E8D57u, W0 = 0x9E3779B9u;
    const uint32_t k0 = (uint32_t)seed, k1 = (uint32_t)(seed >> 32);
    const uint32_t lane = threadIdx.x, mask32 = vector_copy((uint32_t)smask), a = vector_copy((uint32_t)A);
    constexpr uint32_t per = S64 ? 2 : 4;
#pragma unroll
    for (int r = 0; r < RM; ++r) {
        const uint64_t i = rb * (64ull * RM) + (uint64_t)r * 64 + lane;
        const bool ok = !CHECK || i < nwords;
        const uint64_t w = A * i;
        const uint32_t tag = S64 ? kMcTag ^ (uint32_t)(i >> 32) : kMcTag;
        const uint64_t row1 = (uint64_t)M1 * (uint32_t)i;  // round 0
        const uint64_t row2 = (uint64_t)M0 * ((uint32_t)(row1 >> 32) ^ (uint32_t)(j0 / per >> 32) ^ k0);  // round 1
        uint32_t e0 = (uint32_t)row1 ^ keys.a[1], e2 = (uint32_t)(row2 >> 32) ^ keys.b[1],
                 e3 = (uint32_t)row2 ^ keys.b[2];
        asm("" : "+v"(e0), "+v"(e2), "+v"(e3));  // or they are taken apart again in the loop
        const uint64_t jb = CHECK ? jlo / per * per : j0;
        uint64_t q0 = (uint64_t)M0 * (uint32_t)(jb / per);
        for (uint32_t left = uniform32((uint32_t)((j1 - jb + per - 1) / per)), o = 0; left; --left, o += per, q0 += M0) {
            const uint64_t j = jb + o;
            const uint64_t q1 = (uint64_t)M1 * ((uint32_t)(q0 >> 32) ^ tag ^ k1);
            const uint64_t p0 = (uint64_t)keys.m0 * (e0 ^ (uint32_t)(q1 >> 32)), p1 = (uint64_t)keys.m1 * (e2 ^ (uint32_t)q0);
            uint32_t c[4] = {(uint32_t)(p1 >> 32) ^ ((uint32_t)q1 ^ (k0 + 2 * W0)), (uint32_t)p1,
                             (uint32_t)(p0 >> 32) ^ e3, (uint32_t)p0};
            philox_rounds<3>(c, keys);
            if (S64) {
#pragma unroll
                for (uint32_t u = 0; u < 2; ++u) {
                    const uint64_t x = ((uint64_t)c[2 * u] | ((uint64_t)c[2 * u + 1] << 32)) & smask;
                    const uint32_t d = (uint32_t)__popcll(w ^ (A * x));
                    lds_inc(lane_col + ((!CHECK || (ok && j + u >= jlo && j + u < j1)) ? d : dummy) * kStride);
                }
            } else {
#pragma unroll
                for (uint32_t u = 0; u < 4; ++u) {
                    const uint32_t x = c[u] & mask32;
                    const uint32_t d = WIDTH == 0   ? (uint32_t)__popc((uint32_t)w ^ (a * x))
                                       : WIDTH == 1 ? (uint32_t)__popcll(w ^ ((uint64_t)a * x))
                                                    : (uint32_t)__popcll(w ^ (A * (uint64_t)x));
                    lds_inc(lane_col + ((!CHECK || (ok && j + u >= jlo && j + u < j1)) ? d : dummy) * kStride);
                }
            }
        }
    }
}

// Item t of segment s (McSegment: samples [j0, j1) with a histogram of its
// own) = (row group of G row blocks, sample chunk): local index t -
// item_begin = rg * chunks + c, chunk c covering [a + c*CJ, a + (c+1)*CJ) of
// [j0, j1), a = j0 rounded down to CJ.  G is chosen on the host so that an
// item holds about 2^18 pairs (one work-queue step per item).  Segments are
// laid out one after the other, so a wave's items stay in one segment for
// long runs; its LDS rows go to the segment's histogram when the segment
// changes.  ONE: the one segment `single`, whose histogram goes to `direct`, in
// place of the device array.
template <bool ONE>
__global__ __launch_bounds__(64) void an_mc_kernel(uint64_t A, uint32_t n, uint64_t seed, uint32_t G,
                                                   uint32_t CJ, uint32_t heads, const McSegment *__restrict__ segs,
                                                   uint32_t nsegs, uint64_t total_items,
                                                   unsigned long long *__restrict__ counter, uint32_t nbins,
                                                   uint32_t lds_rows, const McSegment single,
                                                   const DirectResult direct) {
    extern __shared__ uint32_t lds[];
    if (ONE) direct_start(direct);
    const uint32_t lane = threadIdx.x;
    lds_clear(lds, lds_rows);
    uint32_t *const lane_col = lds + lane;
    const uint32_t dummy = lds_rows - 1;
    const uint64_t nwords = 1ull << n;
    const uint64_t RBlocks = (nwords + 64ull * RM - 1) / (64ull * RM);
    const uint64_t smask = nwords - 1;
    const PhiloxKeys keys = philox_keys(seed);
    // all codewords (A * (2^n - 1)) below 2^32
    const bool w1 = ((unsigned __int128)A * (nwords - 1)) >> 32 == 0;
    const bool s64 = n > 32;
    uint64_t pending = 0;  // increments per lane counter since the last flush (bound)
    uint32_t cur = 0xFFFFFFFFu;  // segment whose counts the LDS rows hold
    auto flush = [&] {
        if (cur != 0xFFFFFFFFu)
            flush_rows(lds, 0, nbins, ONE ? hist_copy(direct.copies, nbins, kHistCopies)
                                          : hist_copy(segs[cur].out, nbins, (uint32_t)segs[cur].out_copies));
    };
    for (uint64_t t = first_item(); t < total_items; t = following_item_of(counter, heads)) {
        uint32_t sg = cur == 0xFFFFFFFFu ? 0 : cur;
        if (!ONE) {
            while (sg + 1 < nsegs && t >= segs[sg + 1].item_begin) ++sg;
            while (t < segs[sg].item_begin) --sg;
            sg = uniform32(sg);
        }
        const McSegment &seg = ONE ? single : segs[sg];
        const uint64_t local = t - seg.item_begin;
        const uint64_t rg = uniform64(local / seg.chunks), c = uniform64(local - rg * seg.chunks);
        const uint64_t j0 = (seg.j0 & ~(uint64_t)(CJ - 1)) + c * CJ;
        const uint64_t jlo = j0 > seg.j0 ? j0 : seg.j0;
        const uint64_t j1 = j0 + CJ < seg.j1 ? j0 + CJ : seg.j1;
        const uint64_t add = (uint64_t)G * RM * (j1 - j0);
        if (sg != cur || pending + add >= 0xFFFFFFFFull) {
            flush();
            cur = sg;
            pending = 0;
        }
        pending += add;
        for (uint32_t g = 0; g < G; ++g) {
            const uint64_t rb = rg * G + g;
            if (rb >= RBlocks) break;
            // whole rows and whole Philox blocks: no masking
            const bool full = (rb + 1) * (64ull * RM) <= nwords && jlo == j0 && (j1 - j0) % (s64 ? 2 : 4) == 0;
            if (s64) {
                if (full)
                    an_mc_item<2, true, false>(lane_col, A, rb, nwords, j0, jlo, j1, smask, seed, keys, dummy);
                else
                    an_mc_item<2, true, true>(lane_col, A, rb, nwords, j0, jlo, j1, smask, seed, keys, dummy);
            } else if (!full) {
                an_mc_item<2, false, true>(lane_col, A, rb, nwords, j0, jlo, j1, smask, seed, keys, dummy);
            } else if (w1) {
                an_mc_item<0, false, false>(lane_col, A, rb, nwords, j0, jlo, j1, smask, seed, keys, dummy);
            } else if (A >> 32 == 0) {
                an_mc_item<1, false, false>(lane_col, A, rb, nwords, j0, jlo, j1, smask, seed, keys, dummy);
            } else {
                an_mc_item<2, false, false>(lane_col, A, rb, nwords, j0, jlo, j1, smask, seed, keys, dummy);
            }
        }
    }
    flush();
    if (ONE) direct_finish(direct, nbins, lds);
}

__global__ __launch_bounds__(256) void batch_begin(unsigned long long *__restrict__ hist, uint32_t entries,
                                                   const DirectResult out) {
    direct_start(out);
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < entries; i += gridDim.x * 256) hist[i] = 0;
}

// One workgroup: the stores that the end clock waits for are its own.
__global__ __launch_bounds__(1024) void batch_end(const unsigned long long *__restrict__ hist, uint32_t entries,
                                                  unsigned long long *__restrict__ host, const DirectResult out) {
    for (uint32_t i = threadIdx.x; i < entries; i += 1024)
        __hip_atomic_store(host + i, hist[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    direct_end(out);
}

// Dynamic LDS of a Hamming wave: the histogram rows (the syndrome tables are
// the kernel's static LDS).
size_t ham_lds_bytes(uint32_t lds_rows) { return (size_t)lds_rows * kStride * sizeof(uint32_t); }

const void *ham_kernel_ptr(bool w64, bool one) {
    if (one)
        return w64 ? reinterpret_cast<const void *>(&ham_kernel<true, true>)
                   : reinterpret_cast<const void *>(&ham_kernel<false, true>);
    return w64 ? reinterpret_cast<const void *>(&ham_kernel<true, false>)
               : reinterpret_cast<const void *>(&ham_kernel<false, false>);
}

// Resident waves per CU (one query per kernel and rows: a property of the
// kernel and of gfx950's CU), 0 if the query fails.
uint32_t ham_per_cu(bool w64, uint32_t lds_rows) {
    static std::atomic<int> cache[2][132];
    if (lds_rows > 131) return 0;
    int n = cache[w64][lds_rows].load(std::memory_order_relaxed);
    if (n > 0) return (uint32_t)n;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, ham_kernel_ptr(w64, false), 64, ham_lds_bytes(lds_rows)) !=
            hipSuccess ||
        n <= 0)
        return 0;
    cache[w64][lds_rows].store(n, std::memory_order_relaxed);
    return (uint32_t)n;
}

}  // namespace

namespace {

// Waves of a launch, and whether a static assignment replaces the queue.
cr_status ham_waves(bool w64, uint64_t total_items, bool allow_static, uint32_t lds_rows, int cus, uint64_t *out) {
    if (lds_rows < 2 || lds_rows > 131) return fail(CR_ERR_INVALID_ARGUMENT, "bad histogram rows %u", lds_rows);
    const uint32_t per_cu = ham_per_cu(w64, lds_rows);
    if (per_cu == 0) return fail(CR_ERR_DEVICE, "occupancy query failed for the Hamming kernel");
    uint64_t waves = (uint64_t)per_cu * cus;
    if (waves > total_items) waves = total_items;
    if (waves == 0) waves = 1;
    if (allow_static && total_items > 0) {
        // static assignment over at most one wave per CU less than the
        // resident capacity, each wave taking the same number of items
        const uint64_t cap = (uint64_t)(per_cu > 1 ? per_cu - 1 : 1) * cus;
        if (waves > cap) waves = cap;
        const uint64_t per = (total_items + waves - 1) / waves;
        waves = (total_items + per - 1) / per;
    }
    *out = waves;
    return CR_OK;
}

cr_status ham_launch(const HamJob *jobs, uint32_t njobs, uint64_t total_items, bool w64, unsigned long long *counter,
                     uint32_t lds_rows, uint64_t waves, const HamJob &single, const DirectResult &out,
                     hipStream_t stream) {
    const HamJob *a_jobs = jobs;
    uint32_t a_nj = njobs, a_rows = lds_rows;
    uint64_t a_items = total_items;
    unsigned long long *a_counter = counter;
    void *args[] = {(void *)&a_jobs, &a_nj, &a_items, &a_counter, &a_rows, (void *)&single, (void *)&out};
    CR_HIP(hipLaunchKernel(ham_kernel_ptr(w64, !jobs), dim3((uint32_t)waves), dim3(64), args, ham_lds_bytes(lds_rows), stream));
    return CR_OK;
}

}  // namespace

cr_status launch_hamming(const HamJob *d_jobs, uint32_t njobs, uint64_t total_items, bool w64,
                         unsigned long long *counter, bool allow_static, uint32_t lds_rows, int cus,
                         hipStream_t stream) {
    uint64_t waves = 0;
    CR_TRY(ham_waves(w64, total_items, allow_static, lds_rows, cus, &waves));
    if (allow_static && total_items > 0) counter = nullptr;
    if (counter) CR_TRY(fill_zero_u64(counter, 1, stream));
    return ham_launch(d_jobs, njobs, total_items, w64, counter, lds_rows, waves, HamJob{}, DirectResult{}, stream);
}

cr_status launch_batch_begin(unsigned long long *hist, uint32_t entries, const DirectResult &out, hipStream_t stream) {
    hipLaunchKernelGGL(batch_begin, dim3((entries + 255) / 256), dim3(256), 0, stream, hist, entries, out);
    CR_HIP(hipGetLastError());
    return CR_OK;
}

cr_status launch_batch_end(const unsigned long long *hist, uint32_t entries, unsigned long long *host,
                           const DirectResult &out, hipStream_t stream) {
    hipLaunchKernelGGL(batch_end, dim3(1), dim3(1024), 0, stream, hist, entries, host, out);
    CR_HIP(hipGetLastError());
    return CR_OK;
}

cr_status launch_hamming_direct(const HamJob &job, bool w64, bool allow_static, uint32_t lds_rows,
                                const DirectResult &out, int cus, hipStream_t stream) {
    uint64_t waves = 0;
    CR_TRY(ham_waves(w64, job.items, allow_static, lds_rows, cus, &waves));
    return ham_launch(nullptr, 1, job.items, w64, allow_static ? nullptr : out.queue, lds_rows, waves, job, out,
                      stream);
}

uint64_t hamming_items(uint64_t count, uint32_t lane_samples) {
    const uint64_t per_item = 64ull * lane_samples;
    return (count + per_item - 1) / per_item;
}

uint32_t hamming_waves_per_cu(uint32_t lds_rows) {
    return std::max(std::max(ham_per_cu(false, lds_rows), ham_per_cu(true, lds_rows)), 1u);
}

cr_status launch_an_mc(uint64_t A, uint32_t n, uint64_t seed, McSegment *segs, uint32_t nsegs, McSegment *d_segs,
                       unsigned long long *counter, uint32_t nbins, int cus, hipStream_t stream, hipEvent_t ev0,
                       hipEvent_t ev1, const DirectResult *direct) {
    const uint32_t lds_rows = nbins + 1;
    if (lds_rows > 66) return fail(CR_ERR_INVALID_ARGUMENT, "bad histogram rows %u", lds_rows);
    if (nsegs == 0) return fail(CR_ERR_INVALID_ARGUMENT, "no sample range");
    if (direct && nsegs != 1) return fail(CR_ERR_INVALID_ARGUMENT, "one launch, %u sample ranges", nsegs);
    const void *k = direct ? reinterpret_cast<const void *>(&an_mc_kernel<true>)
                           : reinterpret_cast<const void *>(&an_mc_kernel<false>);
    const size_t lds = (size_t)lds_rows * kStride * sizeof(uint32_t);
    static std::atomic<int> cache[2][67];
    int per_cu = cache[direct != nullptr][lds_rows].load(std::memory_order_relaxed);
    if (per_cu <= 0) {
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k, 64, lds) != hipSuccess || per_cu <= 0)
            return fail(CR_ERR_DEVICE, "occupancy query failed for the AN Monte Carlo kernel");
        cache[direct != nullptr][lds_rows].store(per_cu, std::memory_order_relaxed);
    }
    const uint64_t RBlocks = ((1ull << n) + 64ull * RM - 1) / (64ull * RM);
    uint64_t total_chunks = 0, longest = 0, samples = 0;
    for (uint32_t s = 0; s < nsegs; ++s) {
        if (segs[s].j1 <= segs[s].j0) return fail(CR_ERR_INVALID_ARGUMENT, "empty sample range");
        longest = std::max(longest, segs[s].j1 - segs[s].j0);
        samples += segs[s].j1 - segs[s].j0;
    }
    const uint64_t resident = (uint64_t)per_cu * cus;
    // Samples per item, and queue heads.  Waves of a CU progress unevenly (the
    // oldest issues first), so a short launch needs some six items a wave, and
    // that many steps of one head would serialize (12.5 ns each): 8 heads, one an
    // XCD.  Longer launches have one, which also evens out the XCDs (with 8
    // heads 4 % slower).  A = 61, calls of 2^8 words x 10000 samples 65 -> 26 us,
    // 2^16 x 1000 78 -> 62 us, 2^16 x 10000 332 -> 285 us (some 15 of it this).
    uint32_t CJ = 16;
    while (CJ < kMaxChunk && (long double)CJ * 6 * resident < (long double)RBlocks * samples) CJ *= 2;
    for (uint32_t s = 0; s < nsegs; ++s) {
        segs[s].chunks = (segs[s].j1 - segs[s].j0 / CJ * CJ + CJ - 1) / CJ;
        total_chunks += segs[s].chunks;
    }
    // row blocks per item: about 2^18 pairs per item (a power of two up to
    // 4096), keeping at least 16 items per resident wave
    const uint64_t chunk = longest < CJ ? longest : CJ;
    uint32_t G = 1;
    while (G < 4096 && (uint64_t)G * 64 * RM * chunk < (1ull << 18) &&
           ((RBlocks + 2 * G - 1) / (2 * G)) * total_chunks >= 16 * resident)
        G *= 2;
    const uint64_t RG = (RBlocks + G - 1) / G;
    uint64_t items = 0;
    for (uint32_t s = 0; s < nsegs; ++s) {
        segs[s].item_begin = items;
        items += RG * segs[s].chunks;
    }
    uint64_t waves = resident;
    if (waves > items) waves = items;
    if (!direct) {
        CR_HIP(hipMemcpyAsync(d_segs, segs, nsegs * sizeof(McSegment), hipMemcpyHostToDevice, stream));
        CR_TRY(fill_zero_u64(counter, kQueues * kQueuePitch, stream));
    }
    if (ev0) CR_HIP(hipEventRecord(ev0, stream));
    uint64_t a_A = A, a_seed = seed, a_items = items;
    uint32_t a_n = n, a_G = G, a_CJ = CJ, a_heads = CJ < kMaxChunk ? kQueues : 1, a_nsegs = nsegs, a_nbins = nbins, a_rows = lds_rows;
    const McSegment *a_segs = direct ? nullptr : d_segs;
    unsigned long long *a_counter = direct ? direct->queue : counter;
    McSegment a_single = segs[0];
    DirectResult a_direct = direct ? *direct : DirectResult{};
    void *args[] = {&a_A, &a_n, &a_seed, &a_G, &a_CJ, &a_heads, &a_segs, &a_nsegs, &a_items, &a_counter, &a_nbins, &a_rows, &a_single,
                    &a_direct};
    CR_HIP(hipLaunchKernel(k, dim3((uint32_t)waves), dim3(64), args, lds, stream));
    if (ev1) CR_HIP(hipEventRecord(ev1, stream));
    return CR_OK;
}

}  // namespace cr
