// Internal declarations shared by the library's translation units.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstdint>
#include <string>
#include <vector>

#include "coding_reliability.h"

namespace cr {

// Records a message for cr_last_error() on this thread and returns s.
cr_status fail(cr_status s, const char *fmt, ...) __attribute__((format(printf, 2, 3)));
void clear_error();

#define CR_HIP(call)                                                                                 \
    do {                                                                                             \
        hipError_t e_ = (call);                                                                      \
        if (e_ != hipSuccess)                                                                        \
            return ::cr::fail(e_ == hipErrorOutOfMemory ? CR_ERR_OUT_OF_MEMORY : CR_ERR_DEVICE,      \
                              "%s failed: %s (%s:%d)", #call, hipGetErrorString(e_), __FILE__,       \
                              __LINE__);                                                             \
    } while (0)

#define CR_TRY(expr)                                                                                 \
    do {                                                                                             \
        cr_status s_ = (expr);                                                                       \
        if (s_ != CR_OK) return s_;                                                                  \
    } while (0)

// Device memory that grows on demand and is freed with its owner.
struct DeviceBuffer {
    void *ptr = nullptr;
    size_t bytes = 0;
    cr_status reserve(size_t want);
    void release();
    template <class T> T *as() const { return static_cast<T *>(ptr); }
};

// Pinned host memory that grows on demand.
struct HostBuffer {
    void *ptr = nullptr;
    size_t bytes = 0;
    cr_status reserve(size_t want);
    void release();
    template <class T> T *as() const { return static_cast<T *>(ptr); }
};

// ---------------------------------------------------------------------------
// Pair-histogram jobs (exhaustive AN and integer-stride grids).
//
// A job is the triangle {0 <= i < j < N} over codewords A*i.  Rows are cut in
// blocks of RB = 64*R words (R codewords per lane held in registers); the
// columns j >= b*RB of row block b are cut at multiples of CW = Q*RB into
// items.  Item (b, c) covers columns [max(c*CW, b*RB), min((c+1)*CW, N)); the
// part below (b+1)*RB is the diagonal block and is masked to j > i.
// ---------------------------------------------------------------------------
enum PairMode : uint32_t {
    kModeW1 = 0,     // all codewords < 2^32: xor + bcnt per pair
    kModeW2Seg = 1,  // 64-bit codewords, column high dword constant over long segments
    kModeWide = 2,   // 64-bit codewords, high dword of every column: matrix instructions
};

struct PairJob {
    uint64_t A;
    uint64_t N;
    uint64_t item_begin;  // global index of the job's first item in this launch
    uint64_t items;       // items of this job in this launch
    uint64_t item_offset; // local index of the first item (a launch may run a slice)
    uint64_t T;           // row blocks
    uint64_t NC;          // column chunks
    unsigned long long *out;  // device histogram, nbins entries, accumulated with atomics
    uint32_t Q;           // chunk width in row blocks
    uint32_t mode;
    uint32_t nbins;       // bins flushed to out
    uint32_t out_copies;  // copies of the histogram at out (power of two; 0 = 1), hist_copy_stride apart
};
static_assert(sizeof(PairJob) == 80, "PairJob layout");

// sum_{x=0}^{b-1} floor(x/Q); Q = 1 (every small job) without a division
__host__ __device__ inline uint64_t pair_floor_sum(uint64_t b, uint64_t Q) {
    if (Q == 1) return b * (b - 1) / 2;
    const uint64_t q = b / Q, r = b - q * Q;
    return Q * (q * (q - (q > 0 ? 1 : 0)) / 2) + r * q;
}
// items of row blocks [0, b)
__host__ __device__ inline uint64_t pair_prefix(uint64_t b, uint64_t NC, uint64_t Q) {
    return b * NC - pair_floor_sum(b, Q);
}

// Single-code launches below this many pairs run with a static assignment
// (about 100 us of work at 9.6e12 pairs/s: the queue's serialized atomics,
// one per item, would cost more than a static assignment's imbalance).
constexpr long double kStaticPairs = 1e9;

// Tuning for one pair job when the caller leaves a knob at 0: enough items
// (about 16 per resident wave) to balance the persistent waves, rows per lane
// large enough to amortise the per-item set-up.
void auto_pair_tuning(uint64_t N, uint32_t resident_waves, uint32_t &R, uint32_t &Q);

// Looks up (once per device, with that device current) the address of the
// allocation-free entry point's file-scope scratch array on `device`.
cr_status noalloc_setup_device(int device);

// Fills job geometry for R rows per lane and chunk width Q (in row blocks).
void pair_job_geometry(PairJob &job, uint32_t R, uint32_t Q);
// Bit length of the largest codeword (N-1)*A, i.e. the highest possible distance.
uint32_t pair_max_distance(uint64_t A, uint64_t N);
// Chooses the kernel mode for a job.
uint32_t pair_mode(uint64_t A, uint64_t N);

struct PairLaunchConfig {
    uint32_t R = 8;
    uint32_t waves = 0;         // 0 = resident capacity of the device
    uint32_t lds_rows = 0;      // histogram rows in LDS (max nbins + 1 dummy row)
    bool wide = false;          // some job has kModeWide
    uint32_t heads = 1;         // work-queue heads (dev::kQueues of them dev::kQueuePitch apart)
    bool zero_counter = true;   // false: the caller cleared the queue head already
    bool allow_static = false;  // a short launch: static assignment of items to waves, no queue
};

// Launches zero-fill + persistent pair kernel on `stream` for the device job
// array d_jobs (njobs entries, item_begin prefix-summed), with `counter`
// (device u64) as the work queue head.  Histograms jobs[i].out are NOT cleared
// here.  Records ev0/ev1 around the pair kernel when non-null.
cr_status launch_pairs(const PairJob *d_jobs, uint32_t njobs, uint64_t total_items,
                       unsigned long long *counter, const PairLaunchConfig &cfg, int cus,
                       hipStream_t stream, hipEvent_t ev0, hipEvent_t ev1);

// Resident single-wave workgroups per CU for the pair kernel with R rows per
// lane and `lds_rows` histogram rows.
uint32_t pair_waves_per_cu(uint32_t R, uint32_t lds_rows, bool wide);

// Pair histogram of a short code in one launch (see short_pairs.hip).
constexpr uint32_t kShortWords = (1u << 16) - 1;
namespace dev {
struct DirectResult;
}
cr_status launch_short_pairs(uint64_t A, uint32_t N, uint32_t nbins, const dev::DirectResult &out, int cus,
                             hipStream_t stream);
// Buffers of a one-launch call on a context, cleared if an earlier call left
// counts in them, and its end: waits, raw[0, need) from pinned memory, zeros
// above, the device time.
cr_status direct_result(cr_context *ctx, dev::DirectResult *r);
cr_status direct_poll(cr_context *ctx, double *kernel_ms);
cr_status direct_wait(cr_context *ctx, uint64_t *raw, uint32_t need, uint32_t nbins, double *kernel_ms);

// Pair histograms of whole codes by bit planes (see sliced_pairs.hip).
struct SlicedJob {
    uint64_t item_begin, items;  // global range of the job's items in the launch
    unsigned long long *out;     // device histogram, nbins entries, accumulated with atomics
    uint32_t A, Ainv, tc;        // odd part, its inverse modulo 2^k, (A * Ainv - 1) >> k
    uint32_t k;                  // word bits, 11 .. 24
    uint32_t planes;             // codeword bits above the low k, at most 16
    uint32_t parts;              // items that share a 64 x 64 block of words: 1, 2, 4, 8 or 16
    uint32_t nbins, out_copies;  // as PairJob's
};
static_assert(sizeof(SlicedJob) == 56, "SlicedJob layout");
// False when (A, num_words) is outside the kernel.
bool sliced_job(uint64_t A, uint64_t num_words, SlicedJob *j);
// Measured pairs per second of a launch that fills the device.
double sliced_rate(const SlicedJob &j);
// Fills parts, items and item_begin of the jobs of one launch, in order.
void sliced_ranges(std::vector<SlicedJob> &jobs, int cus, uint64_t *total_items);
// counter: the work-queue head, zeroed by the caller, or null for a static
// assignment of items to workgroups.
cr_status launch_sliced(const SlicedJob *d_jobs, uint32_t njobs, uint64_t total_items, unsigned long long *counter,
                        int cus, hipStream_t stream);

// One job (its item range set) whose histogram goes to `out` (out_copies: dev::kHistCopies).
cr_status launch_sliced_direct(const SlicedJob &job, uint64_t items, const dev::DirectResult &out, int cus,
                               hipStream_t stream);

// Rectangle histogram rows x column table (see rect_pairs.hip).
struct RectLaunch {
    uint64_t A = 1, row0 = 0, nrows = 0;
    const uint64_t *rows = nullptr;  // device row table, or null for rows A*(row0+i)
    const uint64_t *cols = nullptr;  // device column table
    uint64_t ncols = 0;
    uint32_t mask32 = 0;             // truncate generated rows to 32 bits
    bool w2 = false;                 // some codeword exceeds 32 bits
    uint32_t nbins = 0, first_bin = 0, lds_rows = 0;
};
cr_status launch_rect(const RectLaunch &L, const dev::DirectResult &out, hipStream_t stream, int cus);

// The same histogram over rows A*i, i < 2^n, by recursion over the carries
// (see carry_rows.hip).
struct CarryRowsPlan {
    uint32_t A = 0, z = 0;   // odd part of the multiplier, its trailing zero bits
    uint32_t n = 0;
    uint32_t rows = 0, threads = 0;  // distances in LDS, threads of a workgroup
    size_t lds = 0;
    bool wide = false;       // 64-bit counters
};
// False when the recursion does not apply or the rectangle kernel is estimated
// to be faster; nbins: distances of the words and samples.
bool carry_rows_plan(uint64_t A, uint32_t n, uint64_t ncols, uint32_t nbins, CarryRowsPlan *p);
// Leaves the histogram of all samples, nbins counts, in out.host.
cr_status launch_carry_rows(const CarryRowsPlan &p, const uint64_t *cols, uint32_t ncols, uint32_t nbins,
                            const dev::DirectResult &out, int cus, hipStream_t stream);

// Hamming weight jobs (see hamming.hip).
enum HamSource : uint32_t { kHamStride = 1, kHamList = 2, kHamMc = 3 };
struct HamJob {
    uint64_t first;            // stride offset, or first Monte Carlo sample index
    uint64_t stride;
    uint64_t count;            // samples
    const uint64_t *list;      // device list (kHamList)
    uint64_t seed;
    uint64_t item_begin, items;  // global range of this job in the launch
    uint64_t item_offset;        // local index of the first item (slices)
    unsigned long long *out;   // device weight histogram (nbins entries)
    uint64_t masks[7];         // parity masks truncated to k bits, zero when unused
    uint32_t source, k, stream, nbins;
    uint32_t lane_samples;     // samples per lane per work item (power of two in [16, kHamMaxLaneSamples])
    uint32_t out_copies;       // copies of the histogram at out (power of two; 0 = 1), hist_copy_stride apart
};
static_assert(sizeof(HamJob) == 152, "HamJob layout");
constexpr uint32_t kHamMaxLaneSamples = 4096;
constexpr uint32_t kHamMaxBatch = 4096;  // requests per cr_hamming_weights_batch call

// True when num_words = 2^k and cr_an_pairs_spectral supports (A, k) and is
// estimated at under 80 % of the pair kernel's time (measured rates:
// 2.2e-12 s per transformed element plus about 50 us per call, against
// 9.6e12 pairs/s); *seconds (if not NULL) is the estimate.
bool spectral_preferred(uint64_t A, uint64_t num_words, uint32_t *k, double *seconds = nullptr);

// One exhaustive AN histogram by the code's spectrum, split into batches of
// transforms (see spectral.hip): shape, device buffer and slot sizes.
struct SpectralPlan {
    uint64_t Ao = 0, tc = 0, chunks = 0, per_batch = 0, batches = 0, buffer_bytes = 0, slot_entries = 0;
    uint32_t k = 0, n = 0, nw = 0, Ainv = 0, nslots = 0;
    uint32_t layout = 0;          // kSpectralInt32 / kSpectralInt16Pairs (see spectral.hip)
    double sec_per_element = 0;   // measured device seconds per transformed element
};
// Pass structures of the spectral path: index bits 0-15 (or 0-7 for k <= 16)
// then the rest through an int32 (int16) buffer; or, for k = 17 .. 24 and at
// least two transforms, bits 0 .. k-11 of two transforms at once then the
// last 10 bits, through int16.
constexpr uint32_t kSpectralInt32 = 0, kSpectralInt16Pairs = 1;
// False when (A, k) is outside the spectral path (then the pair kernel applies).
bool spectral_plan(uint64_t A, uint32_t k, int cus, SpectralPlan *p);
// Launches batches [first_batch, first_batch + nbatches) on stream, with X of
// p.buffer_bytes and slots of p.slot_entries uint64 (zeroed before the first).
cr_status spectral_run(const SpectralPlan &p, void *X, unsigned long long *slots, uint64_t first_batch,
                       uint64_t nbatches, hipStream_t stream);
// raw[] (nbins entries, pair-kernel form) from the host copy of the slots.
cr_status spectral_finish(const SpectralPlan &p, const uint64_t *slots, uint64_t *raw, uint32_t nbins);

// One exhaustive AN histogram by recursion over the carries of the product
// (see carry.hip).
struct CarryPlan {
    uint32_t A = 0, Ainv = 0;   // odd part of the multiplier, its inverse modulo 2^32
    uint32_t k = 0, T = 0;      // word bits; low bits that the last kernel takes at once (2^T > A)
    uint32_t hb = 0;            // bits of the largest carry, A - 1
    uint32_t levels = 0;        // k - T
    uint32_t states = 0;        // carry pairs, A^2
    uint32_t nbins = 0;         // distances 0 .. k + hb
    uint64_t table_bytes = 0;   // of each of the two tables
    double seconds = 0;         // estimated time of a call
};
// False when (A, 2^k words) is outside the recursion.
bool carry_plan(uint64_t A, uint32_t k, CarryPlan *p);
// Leaves the distribution over ordered pairs, p.nbins counts, in out.host.
cr_status carry_run(const CarryPlan &p, void *table0, void *table1, const dev::DirectResult &out, int cus,
                    hipStream_t stream);
// raw[] (nbins entries, pair-kernel form) from an ordered-pair histogram of 2^k
// words (`copies` copies of `bins`, dev::hist_copy_stride apart); checks the
// words at distance 0 and the total of 4^k.
cr_status carry_finish(uint32_t k, uint32_t bins, const uint64_t *hist, uint32_t copies, uint64_t *raw,
                       uint32_t nbins);

// The same for any word count, odd parts below 1024 (see carry_ragged.hip).
struct CarryRaggedPlan {
    uint32_t A = 0, N = 0;      // odd part of the multiplier, words
    uint32_t T = 0;             // 2^T > A, at least 7
    uint32_t levels = 0;        // the highest bit of N
    uint32_t states = 0;        // carry pairs, A^2
    uint32_t tail = 0;          // words paired one by one
    uint32_t nbins = 0;
    uint64_t table_bytes = 0;   // of each of the two tables
    double seconds = 0;         // estimated time of a call
};
bool carry_ragged_plan(uint64_t A, uint64_t num_words, CarryRaggedPlan *p);
// Leaves the distribution over ordered pairs, p.nbins counts, in out.host.
cr_status carry_ragged_run(const CarryRaggedPlan &p, void *table0, void *table1, const dev::DirectResult &out, int cus,
                           hipStream_t stream);
// raw[] (nbins entries, pair-kernel form) from `bins` counts of ordered pairs of
// `words` words; checks the words at distance 0 and the total.
cr_status ordered_finish(uint64_t words, uint32_t bins, const uint64_t *hist, uint64_t *raw, uint32_t nbins);

// The same recursion for long multipliers, by tiles of carry pairs with four
// levels a kernel (see carry_tiles.hip).
struct CarryTilesPlan {
    uint32_t A = 0, k = 0;
    uint32_t F = 0;             // levels of the second kernel, 0 .. 4
    uint32_t T = 0;             // low bits taken pair by pair, k - 4 - F
    uint32_t hb = 0, nbins = 0;
    uint64_t table_bytes = 0, hist_entries = 0;
    double seconds = 0;         // estimated time of a call
};
bool carry_tiles_plan(uint64_t A, uint32_t k, CarryTilesPlan *p);
cr_status carry_tiles_run(const CarryTilesPlan &p, void *table, unsigned long long *hist, int cus,
                          hipStream_t stream);

// The methods of cr_an_pairs for a code, by their estimated times: the fastest,
// then those that take its place when device memory for its tables lacks.  The
// last one takes no tables.
enum PairsMethod : uint32_t { kByPairs, kByShort, kByPlanes, kBySpectrum, kByCarry, kByTiles, kByBlocks };
struct PairsPlan {
    uint32_t methods = 0;
    uint32_t method[5];
    uint32_t k = 0;  // kBySpectrum: 2^k words
    SlicedJob sliced;
    CarryPlan carry;
    CarryTilesPlan tiles;
    CarryRaggedPlan ragged;
};
void pairs_plan(uint64_t A, uint64_t num_words, PairsPlan *p);

// Weight histogram of consecutive data words, bit by bit of their bounds (see
// hamming_range.hip).
struct HamRange {
    unsigned long long *out;  // device histogram, nbins entries (written, not added to)
    uint32_t r, nbins;
    uint32_t steps;       // of two data bits, from the top
    uint32_t start_bits;  // 1 for an odd width, whose top bit the start entries include
    struct Start {
        uint64_t weight;
        uint32_t at, reserved;  // at: (popcount << r) + parity bits
    } start[4];
    struct Step {
        uint16_t col[2];  // parity bits of the step's upper and lower data bit
        struct {
            uint16_t at;
            int16_t sign;
        } enter[6];  // words that leave the range's start (-1) or end (+1) in this step
    } step[32];
};
// The words [first, first + count) modulo 2^k; job->r is set.
void ham_range_job(uint64_t first, uint64_t count, uint32_t k, const uint64_t masks[7], HamRange *job);
// The jobs of a device array, or (single) one whose histogram goes to out.host;
// the largest width and parity bits among them.
cr_status launch_ham_ranges(const HamRange *d_jobs, uint32_t njobs, const HamRange *single, uint32_t max_k,
                            uint32_t max_r, const dev::DirectResult &out, hipStream_t stream);

// Parity masks of the (N,k) extended Hamming codes, truncated to k bits;
// returns the number of non-overall parity bits.
uint32_t hamming_masks(uint32_t k, uint64_t masks[7]);
// Work items of a job of `count` samples at lane_samples per lane (64 lanes).
uint64_t hamming_items(uint64_t count, uint32_t lane_samples);
// Waves per CU of the Hamming kernel (the larger of the 32- and 64-bit forms).
uint32_t hamming_waves_per_cu(uint32_t lds_rows);
// counter: the work-queue head (zeroed here).  allow_static: a short launch
// of equal items, run with a static assignment of items to waves instead of
// the queue.
cr_status launch_hamming(const HamJob *d_jobs, uint32_t njobs, uint64_t total_items, bool w64,
                         unsigned long long *counter, bool allow_static, uint32_t lds_rows, int cus,
                         hipStream_t stream);
// The first and the last launch of a small batch: `entries` counters cleared and
// the start clock; the counters copied to pinned memory and the end clock.
cr_status launch_batch_begin(unsigned long long *hist, uint32_t entries, const dev::DirectResult &out,
                             hipStream_t stream);
cr_status launch_batch_end(const unsigned long long *hist, uint32_t entries, unsigned long long *host,
                           const dev::DirectResult &out, hipStream_t stream);
// One job whose histogram goes to `out` (out_copies: dev::kHistCopies).
cr_status launch_hamming_direct(const HamJob &job, bool w64, bool allow_static, uint32_t lds_rows,
                                const dev::DirectResult &out, int cus, hipStream_t stream);
// A sample range of an AN Monte Carlo launch and its histogram: the pairs
// (word i, sample j) for every word i and j0 <= j < j1 (j0 < j1).
struct McSegment {
    uint64_t j0, j1;
    uint64_t item_begin;      // first work item of the range (set by launch_an_mc)
    uint64_t chunks;          // sample chunks of the range (set by launch_an_mc)
    unsigned long long *out;  // device histogram (zeroed by the caller), out_copies copies of it
    uint64_t out_copies;
};
constexpr uint32_t kMcMaxRanges = 64;  // sample ranges per AN Monte Carlo launch
// segs (host, nsegs entries, kept alive until the stream is synchronized) is
// completed and copied to d_segs; counter holds the work-queue heads (zeroed here).
// direct (one segment): its histogram goes there, nothing is copied or zeroed,
// and d_segs, counter and the events are not used.
cr_status launch_an_mc(uint64_t A, uint32_t n, uint64_t seed, McSegment *segs, uint32_t nsegs, McSegment *d_segs,
                       unsigned long long *counter, uint32_t nbins, int cus, hipStream_t stream, hipEvent_t ev0,
                       hipEvent_t ev1, const dev::DirectResult *direct);

// Zero-fills n 64-bit words on stream (a kernel, so it may be captured in graphs).
cr_status fill_zero_u64(unsigned long long *p, size_t n, hipStream_t stream);

}  // namespace cr

struct cr_context {
    int device = 0;
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    int cus = 0;
    int clock_mhz = 0;
    int wall_khz = 0;          // rate of the device's constant clock
    uint64_t hbm = 0;
    char name[64] = {0};
    char arch[32] = {0};
    cr::DeviceBuffer jobs;     // PairJob array
    cr::DeviceBuffer counters; // work-queue heads
    cr::DeviceBuffer hist;     // histograms
    cr::DeviceBuffer direct;   // histogram copies, queue heads and tickets of one-launch calls
    bool direct_clean = false; // they are zero: the last such call came to its end
    cr::DeviceBuffer table_a;  // row / sample tables
    cr::DeviceBuffer table_b;
    cr::HostBuffer host;       // pinned staging
};
