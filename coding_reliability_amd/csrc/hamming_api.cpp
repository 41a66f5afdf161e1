// Host side of the Extended Hamming and AN Monte Carlo entry points.
#include <algorithm>
#include <cstring>
#include <vector>

#include "cr_device.h"
#include "cr_internal.h"

namespace cr {

// The reference's (39,32) parity masks (distance_distribution/src/hamming.h:54-64)
// are the low halves of the (72,64) patterns of legacy/Hamming/ExtHamming64.hpp:31-37;
// one table truncated to the data width serves every k.
static const uint64_t kHamPatterns[7] = {
    0xAB55555556AAAD5Bull, 0xCD9999999B33366Dull, 0x78F1E1E1E3C3C78Eull, 0x01FE01FE03FC07F0ull,
    0x01FFFE0003FFF800ull, 0x01FFFFFFFC000000ull, 0xFE00000000000000ull};

uint32_t hamming_masks(uint32_t k, uint64_t masks[7]) {
    const uint64_t dm = k >= 64 ? ~0ull : ((1ull << k) - 1);
    uint32_t r = 0;
    for (int t = 0; t < 7; ++t) {
        masks[t] = kHamPatterns[t] & dm;
        if (masks[t]) ++r;
    }
    return r;
}

}  // namespace cr

using namespace cr;

extern "C" uint32_t cr_hamming_parity_bits(uint32_t k) {
    uint64_t m[7];
    return hamming_masks(k, m);
}

namespace {

// The weight bins of a request, after its checks.
cr_status ham_check(const cr_ham_request *req, uint32_t nbins, uint32_t *need, uint32_t *parity, uint64_t masks[7]) {
    if (req->k < 1 || req->k > 64) return fail(CR_ERR_INVALID_ARGUMENT, "k=%u outside [1, 64]", req->k);
    if (req->source > CR_HAM_MC) return fail(CR_ERR_INVALID_ARGUMENT, "unknown source %u", req->source);
    if (req->source == CR_HAM_LIST && req->count && !req->list)
        return fail(CR_ERR_INVALID_ARGUMENT, "list source without a list");
    const uint32_t per = req->k <= 32 ? 4 : 2;
    if (req->source == CR_HAM_MC && req->first % per)
        return fail(CR_ERR_INVALID_ARGUMENT, "Monte Carlo first sample must be a multiple of %u", per);
    *parity = hamming_masks(req->k, masks);
    *need = req->k + *parity + 1;  // weights 0..k+r
    if (nbins < *need) return fail(CR_ERR_INVALID_ARGUMENT, "nbins=%u but weights reach %u", nbins, *need - 1);
    return CR_OK;
}

HamRange ham_range(const cr_ham_request *req, uint32_t need, uint32_t parity, const uint64_t masks[7]) {
    HamRange job{};
    job.r = parity;
    job.nbins = need;
    ham_range_job(req->first, req->count, req->k, masks, &job);
    return job;
}

// Measured rates (words/s, launches of 2^30 words; 64-bit strides reach 1.2e12 there
// and this at 2^27): 32-bit stride 2.5e12, 64-bit 0.9e12, Monte Carlo 1.9e12 /
// 0.87e12, lists about half the stride rates.
double ham_rate(const cr_ham_request *req) {
    if (req->source == CR_HAM_MC) return req->k > 32 ? 0.87e12 : 1.9e12;
    return (req->k > 32 ? 0.9e12 : 2.5e12) * (req->source == CR_HAM_LIST ? 0.5 : 1.0);
}

// A job and its work assignment in a launch of `waves` resident waves.  The
// queue balances waves that advance at different rates (a static assignment
// measured about 25 % slower on launches of 0.5 ms and more), but each queue
// step is a device-scope atomic on one counter, serialized at about 12.5 ns, one
// per item plus one per wave: 40-150 us per launch.  Launches estimated below
// kShortLaunch of work therefore run with a static assignment (calls of 2.1e8
// 32-bit stride words 124 us with it, 120 with the queue; of 8e7 64-bit Monte
// Carlo words 176 and 148).
constexpr double kShortLaunch = 82e-6;
HamJob ham_job(const cr_ham_request *req, uint32_t need, const uint64_t masks[7], bool short_launch, uint64_t waves) {
    HamJob job{};
    memcpy(job.masks, masks, sizeof(job.masks));
    job.first = req->first;
    job.stride = req->stride;
    job.count = req->count;
    job.seed = req->seed;
    job.source = req->source;
    job.k = req->k;
    job.stream = req->stream;
    job.nbins = need;
    // items of 64 x spl words, spl the smallest power of two in [16,
    // kHamMaxLaneSamples] that gives at most 8 items per resident wave for a
    // static assignment or 32 for the queue (the last items set the launch's
    // tail: with at most 4 per wave a 2^30-word (72,64) Monte Carlo launch ran
    // 20 % below the rate of 2^34 words), and for the queue at least rate/8e7
    // words per item (the counter's 8e7 items/s)
    const uint64_t per_wave = short_launch ? 8 : 32;
    const uint64_t want = (job.count + 64 * per_wave * waves - 1) / (64 * per_wave * waves);
    const double min_words = short_launch ? 0.0 : ham_rate(req) / 8e7;
    uint64_t spl = 16;
    while ((spl < want || 64.0 * (double)spl < min_words) && spl < kHamMaxLaneSamples) spl *= 2;
    job.lane_samples = (uint32_t)spl;
    job.items = hamming_items(job.count, job.lane_samples);
    // dev::kHistCopies line-aligned copies of each histogram, summed at the end
    job.out_copies = dev::kHistCopies;
    return job;
}

// Ranges as the grids of stride 1 that they are, word by word, where a few words
// take less time than the launch of the recursion over their bits: in a launch
// of their width that is there anyway, in calls that are no small batch in
// either way, and from k = 58 on, where the recursion takes 25 to 29 us.  Measured
// beside 2^20 Monte Carlo words of the same width: 1000 words of k = 64 39 us for
// 70, of k = 57 44 for 62, of k = 32 30 for 43; four ranges of 2^20 words 90 us for
// 74 at k = 64, 60 for 51 at k = 20.
constexpr double kWordsSeconds = 1.25e-6;  // of all of them, by ham_rate
constexpr uint32_t kWordsMinK = 58;
constexpr uint32_t kWordRanges = 4;       // eight: 0.85 to 1.22 of the recursion's time
cr_ham_request as_words(const cr_ham_request *range) {
    cr_ham_request r = *range;
    r.source = CR_HAM_STRIDE;
    r.stride = 1;
    return r;
}

// Counters that one workgroup copies in a few us: of six requests of k = 64, ten of k = 32.
constexpr uint64_t kSmallBatch = 16384;

// One request in one launch.
cr_status hamming_single(cr_context *ctx, const cr_ham_request *req, uint64_t *hist, uint32_t nbins,
                         double *kernel_ms) {
    if (!ctx || !req || !hist) return fail(CR_ERR_INVALID_ARGUMENT, "NULL argument");
    uint32_t need = 0, parity = 0;
    uint64_t masks[7];
    CR_TRY(ham_check(req, nbins, &need, &parity, masks));
    CR_HIP(hipSetDevice(ctx->device));
    if (req->count == 0) {
        memset(hist, 0, nbins * sizeof(uint64_t));
        if (kernel_ms) *kernel_ms = 0;
        return CR_OK;
    }
    dev::DirectResult out;
    cr_ham_request words;
    if (req->source == CR_HAM_RANGE && req->k >= kWordsMinK &&
        (double)req->count / ham_rate(req) < kWordsSeconds) {
        words = as_words(req);
        req = &words;
    }
    if (req->source == CR_HAM_RANGE) {
        CR_TRY(direct_result(ctx, &out));
        const HamRange job = ham_range(req, need, parity, masks);
        CR_TRY(launch_ham_ranges(nullptr, 1, &job, req->k, parity, out, ctx->stream));
        return direct_wait(ctx, hist, need, nbins, kernel_ms);
    }
    const bool short_launch = (double)req->count / ham_rate(req) < kShortLaunch;
    const uint32_t rows = need + 1;
    HamJob job = ham_job(req, need, masks, short_launch, (uint64_t)hamming_waves_per_cu(rows) * ctx->cus);
    if (req->source == CR_HAM_LIST) {
        CR_TRY(ctx->table_a.reserve(req->count * sizeof(uint64_t)));
        CR_HIP(hipMemcpyAsync(ctx->table_a.ptr, req->list, req->count * sizeof(uint64_t), hipMemcpyHostToDevice,
                              ctx->stream));
        job.list = ctx->table_a.as<uint64_t>();
    }
    CR_TRY(direct_result(ctx, &out));
    job.out = out.copies;
    CR_TRY(launch_hamming_direct(job, req->k > 32, short_launch, rows, out, ctx->cus, ctx->stream));
    return direct_wait(ctx, hist, need, nbins, kernel_ms);
}

// Requests [0, n): ranges as the workgroups of one launch (few short ones as
// Hamming jobs, see kWordsSeconds), the others as one Hamming job each, those of
// 32-bit words in one launch, those of 64-bit words (k > 32) in another on the
// same stream; requests without samples launch nothing.  hists[i * nbins + b] is
// request i's count of weight b.
cr_status hamming_run(cr_context *ctx, const cr_ham_request *reqs, uint32_t n, uint64_t *hists, uint32_t nbins,
                      double *kernel_ms) {
    if (!ctx || !reqs || !hists) return fail(CR_ERR_INVALID_ARGUMENT, "NULL argument");
    if (n == 0 || n > kHamMaxBatch)
        return fail(CR_ERR_INVALID_ARGUMENT, "%u requests outside [1, %u]", n, kHamMaxBatch);
    if (n == 1) return hamming_single(ctx, reqs, hists, nbins, kernel_ms);
    struct Pending {
        uint32_t index, need, parity;
        uint64_t masks[7];
    };
    struct Launch {
        std::vector<Pending> requests;
        std::vector<HamJob> jobs;
        double est_s = 0;
        uint32_t rows = 2;
        uint64_t items = 0;
        bool short_launch = false;
        void add(const cr_ham_request *req, const Pending &p) {
            est_s += (double)req->count / ham_rate(req);
            rows = std::max(rows, p.need + 1);
            requests.push_back(p);
        }
    } launches[2];
    std::vector<Pending> range_requests;
    std::vector<HamRange> ranges;
    uint32_t range_k = 0, range_r = 0;
    struct Result {
        uint32_t index, need, copies;
        uint64_t at;
    };
    std::vector<Result> results, range_results;
    uint64_t list_words = 0, entries = 0;
    uint64_t job_entries = 0, range_entries = 0;  // counters of the jobs, of the ranges in one copy
    auto job_counters = [](const Pending &p) { return dev::hist_copy_stride(p.need) * dev::kHistCopies; };
    for (uint32_t q = 0; q < n; ++q) {
        const cr_ham_request *req = reqs + q;
        Pending p{q, 0, 0, {}};
        CR_TRY(ham_check(req, nbins, &p.need, &p.parity, p.masks));
        if (req->count == 0) continue;
        if (req->source == CR_HAM_RANGE) {
            range_requests.push_back(p);
            range_entries += dev::hist_copy_stride(p.need);
            continue;
        }
        if (req->source == CR_HAM_LIST) list_words += req->count;
        launches[req->k > 32].add(req, p);
        job_entries += job_counters(p);
    }
    // the ranges all one way or the other: the recursion's launch would stay for one
    double range_s = 0;
    bool joined = true, longest = true;  // launches of their widths are there; k of kWordsMinK and more
    uint64_t word_entries = job_entries;
    for (const Pending &p : range_requests) {
        const cr_ham_request *req = reqs + p.index;
        range_s += (double)req->count / ham_rate(req);
        joined = joined && !launches[req->k > 32].requests.empty();
        longest = longest && req->k >= kWordsMinK;
        word_entries += job_counters(p);
    }
    const bool words = range_requests.size() <= kWordRanges && range_s < kWordsSeconds &&
                       (longest || job_entries + range_entries > kSmallBatch ||
                        (joined && word_entries <= kSmallBatch));
    for (const Pending &p : range_requests) {
        const cr_ham_request *req = reqs + p.index;
        if (words) {
            launches[req->k > 32].add(req, p);
            continue;
        }
        ranges.push_back(ham_range(req, p.need, p.parity, p.masks));
        range_k = std::max(range_k, req->k);
        range_r = std::max(range_r, p.parity);
        range_results.push_back({p.index, p.need, 1, 0});
    }
    CR_HIP(hipSetDevice(ctx->device));
    memset(hists, 0, (size_t)n * nbins * sizeof(uint64_t));
    if (kernel_ms) *kernel_ms = 0;
    if (launches[0].requests.empty() && launches[1].requests.empty() && ranges.empty()) return CR_OK;
    if (list_words) CR_TRY(ctx->table_a.reserve(list_words * sizeof(uint64_t)));
    uint64_t list_at = 0;
    for (Launch &L : launches) {
        L.short_launch = L.est_s < kShortLaunch;
        const uint64_t waves = (uint64_t)hamming_waves_per_cu(L.rows) * ctx->cus;
        for (const Pending &p : L.requests) {
            cr_ham_request words_of;
            const cr_ham_request *req = reqs + p.index;
            if (req->source == CR_HAM_RANGE) {
                words_of = as_words(req);
                req = &words_of;
            }
            HamJob job = ham_job(req, p.need, p.masks, L.short_launch, waves);
            job.item_begin = L.items;
            L.items += job.items;
            if (job.source == kHamList) {
                CR_HIP(hipMemcpyAsync(ctx->table_a.as<uint64_t>() + list_at, req->list, req->count * sizeof(uint64_t),
                                      hipMemcpyHostToDevice, ctx->stream));
                job.list = ctx->table_a.as<uint64_t>() + list_at;
                list_at += req->count;
            }
            results.push_back({p.index, p.need, job.out_copies, entries});
            entries += dev::hist_copy_stride(p.need) * job.out_copies;
            L.jobs.push_back(job);
        }
    }
    for (Result &r : range_results) {
        r.at = entries;
        entries += dev::hist_copy_stride(r.need);
    }
    const size_t njobs = launches[0].jobs.size() + launches[1].jobs.size();
    const size_t job_bytes = njobs * sizeof(HamJob), range_bytes = ranges.size() * sizeof(HamRange);
    CR_TRY(ctx->hist.reserve(entries * sizeof(uint64_t)));
    CR_TRY(ctx->counters.reserve(2 * sizeof(uint64_t)));
    CR_TRY(ctx->jobs.reserve(job_bytes + range_bytes));
    unsigned long long *hist = ctx->hist.as<unsigned long long>();
    std::vector<HamJob> all;
    all.reserve(njobs);
    for (Launch &L : launches)
        for (HamJob &job : L.jobs) {
            job.out = hist + results[all.size()].at;
            all.push_back(job);
        }
    for (size_t j = 0; j < ranges.size(); ++j) ranges[j].out = hist + range_results[j].at;
    // few requests: the counters come back as one-launch calls' do, without the
    // copy, the events and the runtime's wait (the (39,32) stride grid of 2^20
    // words beside one of 2^20 Monte Carlo words: 43 -> 31 us)
    constexpr uint32_t kHeader = dev::kDirectBins + 2;
    const bool small = entries <= kSmallBatch;
    CR_TRY(ctx->host.reserve((kHeader + entries) * sizeof(uint64_t)));
    dev::DirectResult out;
    if (small) {
        CR_TRY(direct_result(ctx, &out));
        CR_TRY(launch_batch_begin(hist, (uint32_t)entries, out, ctx->stream));
    } else {
        CR_TRY(fill_zero_u64(hist, entries, ctx->stream));
    }
    if (njobs) CR_HIP(hipMemcpyAsync(ctx->jobs.ptr, all.data(), job_bytes, hipMemcpyHostToDevice, ctx->stream));
    HamRange *d_ranges = reinterpret_cast<HamRange *>(ctx->jobs.as<char>() + job_bytes);
    if (!ranges.empty())
        CR_HIP(hipMemcpyAsync(d_ranges, ranges.data(), range_bytes, hipMemcpyHostToDevice, ctx->stream));
    // HIP events before the first launch and after the last
    if (kernel_ms && !small) CR_HIP(hipEventRecord(ctx->ev0, ctx->stream));
    if (!ranges.empty())
        CR_TRY(launch_ham_ranges(d_ranges, (uint32_t)ranges.size(), nullptr, range_k, range_r, dev::DirectResult{},
                                 ctx->stream));
    for (int w = 0; w < 2; ++w) {
        const Launch &L = launches[w];
        if (L.jobs.empty()) continue;
        CR_TRY(launch_hamming(ctx->jobs.as<HamJob>() + (w ? launches[0].jobs.size() : 0), (uint32_t)L.jobs.size(),
                              L.items, w == 1, ctx->counters.as<unsigned long long>() + w, L.short_launch, L.rows,
                              ctx->cus, ctx->stream));
    }
    uint64_t *const copies = ctx->host.as<uint64_t>() + kHeader;
    if (small) {
        CR_TRY(launch_batch_end(hist, (uint32_t)entries, reinterpret_cast<unsigned long long *>(copies), out,
                                ctx->stream));
        CR_TRY(direct_poll(ctx, kernel_ms));
    } else {
        if (kernel_ms) CR_HIP(hipEventRecord(ctx->ev1, ctx->stream));
        CR_HIP(hipMemcpyAsync(copies, hist, entries * sizeof(uint64_t), hipMemcpyDeviceToHost, ctx->stream));
        CR_HIP(hipStreamSynchronize(ctx->stream));
    }
    results.insert(results.end(), range_results.begin(), range_results.end());
    for (const Result &r : results) {
        uint64_t *h = hists + (uint64_t)r.index * nbins;
        for (uint32_t c = 0; c < r.copies; ++c)
            for (uint32_t b = 0; b < r.need; ++b) h[b] += copies[r.at + c * dev::hist_copy_stride(r.need) + b];
    }
    if (kernel_ms && !small) {
        float ms = 0;
        CR_HIP(hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1));
        *kernel_ms = ms;
    }
    return CR_OK;
}

}  // namespace

extern "C" cr_status cr_hamming_weights(cr_context *ctx, const cr_ham_request *req, uint64_t *hist, uint32_t nbins,
                                        double *kernel_ms) {
    clear_error();
    return hamming_run(ctx, req, 1, hist, nbins, kernel_ms);
}

extern "C" cr_status cr_hamming_weights_batch(cr_context *ctx, const cr_ham_request *reqs, uint32_t n,
                                              uint64_t *hists, uint32_t nbins, double *kernel_ms) {
    clear_error();
    return hamming_run(ctx, reqs, n, hists, nbins, kernel_ms);
}

extern "C" cr_status cr_hamming_report(uint32_t k, const uint64_t *weights, int with_1bit, uint64_t *out_u128) {
    clear_error();
    if (!weights || !out_u128) return fail(CR_ERR_INVALID_ARGUMENT, "NULL argument");
    if (k < 1 || k > 64) return fail(CR_ERR_INVALID_ARGUMENT, "k=%u outside [1, 64]", k);
    if (k + cr_hamming_parity_bits(k) + 1 > 121) return fail(CR_ERR_UNSUPPORTED, "codeword too long");
    const uint32_t N = k + cr_hamming_parity_bits(k) + 1;  // codeword bits incl. overall parity
    const uint32_t cc = N + 1;
    std::vector<unsigned __int128> c(cc, 0);
    // hamming.cu:183-208
    c[0] = (unsigned __int128)1 << k;
    c[1] = with_1bit ? ((unsigned __int128)1 << k) * N : 0;
    c[2] = 0;
    for (uint32_t i = 4; i < cc; i += 2) {
        c[i] = (unsigned __int128)weights[i] + weights[i - 1];
        c[i - 1] = 0;
    }
    if (with_1bit)
        for (uint32_t i = 3; i < cc; i += 2)
            c[i] = i + 1 < cc ? (unsigned __int128)(i + 1) * c[i + 1] + (unsigned __int128)(N - i + 1) * c[i - 1]
                              : (unsigned __int128)(N - i + 1) * c[i - 1];
    for (uint32_t i = 3; i < cc; ++i) {
        if (c[i] >> (128 - k))
            return fail(CR_ERR_UNSUPPORTED, "reported count of weight %u exceeds 128 bits at k=%u", i, k);
        c[i] <<= k;
    }
    for (uint32_t i = 0; i < cc; ++i) {
        out_u128[2 * i] = (uint64_t)c[i];
        out_u128[2 * i + 1] = (uint64_t)(c[i] >> 64);
    }
    return CR_OK;
}

namespace {

// Histograms of the sample ranges [bounds[i], bounds[i+1]), i < count, in one
// launch: hists[i * nbins + b].  Empty ranges stay zero.
cr_status an_mc_ranges(cr_context *ctx, uint64_t A, uint32_t n, const uint64_t *bounds, uint32_t count,
                       uint64_t seed, uint64_t *hists, uint32_t nbins, double *kernel_ms) {
    if (!ctx || !hists || !bounds) return fail(CR_ERR_INVALID_ARGUMENT, "NULL argument");
    if (A == 0) return fail(CR_ERR_INVALID_ARGUMENT, "A must be >= 1");
    if (n < 1 || n > 63) return fail(CR_ERR_UNSUPPORTED, "AN Monte Carlo supports 1 <= n <= 63 (got %u)", n);
    if ((unsigned __int128)A * ((1ull << n) - 1) >> 64)
        return fail(CR_ERR_UNSUPPORTED, "codewords A*(2^n-1) exceed 64 bits");
    if (count < 1 || count > kMcMaxRanges)
        return fail(CR_ERR_INVALID_ARGUMENT, "%u sample ranges outside [1, %u]", count, kMcMaxRanges);
    for (uint32_t i = 0; i < count; ++i)
        if (bounds[i + 1] < bounds[i]) return fail(CR_ERR_INVALID_ARGUMENT, "sample bounds decrease at %u", i + 1);
    uint32_t bits = 0;
    for (unsigned __int128 x = (unsigned __int128)A * ((1ull << n) - 1); x; x >>= 1) ++bits;
    const uint32_t need = bits + 1;
    if (nbins < need) return fail(CR_ERR_INVALID_ARGUMENT, "nbins=%u but distances reach %u", nbins, need - 1);
    CR_HIP(hipSetDevice(ctx->device));
    if (count == 1 && bounds[1] > bounds[0]) {
        dev::DirectResult direct;
        CR_TRY(direct_result(ctx, &direct));
        McSegment one{bounds[0], bounds[1], 0, 0, nullptr, 1};
        CR_TRY(launch_an_mc(A, n, seed, &one, 1, nullptr, nullptr, need, ctx->cus, ctx->stream, nullptr, nullptr,
                            &direct));
        return direct_wait(ctx, hists, need, nbins, kernel_ms);
    }
    memset(hists, 0, (size_t)count * nbins * sizeof(uint64_t));
    if (kernel_ms) *kernel_ms = 0;
    // copies of each histogram, 64 in all: a short launch is many waves that flush
    // at about the same time, and one histogram serializes their atomics (2^12
    // words x 18151 samples in two ranges 231 us with one copy, 81 with 32)
    uint32_t copies = dev::kHistCopies;
    while (copies > 1 && copies * count > 64) copies /= 2;
    const uint64_t stride = dev::hist_copy_stride(need);
    const uint64_t entries = (uint64_t)count * copies * stride;
    CR_TRY(ctx->hist.reserve(entries * sizeof(uint64_t)));
    CR_TRY(ctx->counters.reserve(dev::kQueues * dev::kQueuePitch * sizeof(uint64_t)));
    CR_TRY(ctx->jobs.reserve(count * sizeof(McSegment)));
    unsigned long long *out = ctx->hist.as<unsigned long long>();
    std::vector<McSegment> segs;
    for (uint32_t i = 0; i < count; ++i)
        if (bounds[i + 1] > bounds[i]) segs.push_back({bounds[i], bounds[i + 1], 0, 0, out + i * copies * stride, copies});
    if (segs.empty()) return CR_OK;
    CR_TRY(fill_zero_u64(out, entries, ctx->stream));
    CR_TRY(launch_an_mc(A, n, seed, segs.data(), (uint32_t)segs.size(), ctx->jobs.as<McSegment>(),
                        ctx->counters.as<unsigned long long>(), need, ctx->cus, ctx->stream,
                        kernel_ms ? ctx->ev0 : nullptr, kernel_ms ? ctx->ev1 : nullptr, nullptr));
    CR_TRY(ctx->host.reserve(entries * sizeof(uint64_t)));
    CR_HIP(hipMemcpyAsync(ctx->host.ptr, out, entries * sizeof(uint64_t), hipMemcpyDeviceToHost, ctx->stream));
    CR_HIP(hipStreamSynchronize(ctx->stream));
    const uint64_t *h = ctx->host.as<uint64_t>();
    for (uint32_t i = 0; i < count; ++i)
        for (uint32_t c = 0; c < copies; ++c, h += stride)
            for (uint32_t b = 0; b < need; ++b) hists[(uint64_t)i * nbins + b] += h[b];
    if (kernel_ms) {
        float ms = 0;
        CR_HIP(hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1));
        *kernel_ms = ms;
    }
    return CR_OK;
}

}  // namespace

extern "C" cr_status cr_an_mc(cr_context *ctx, uint64_t A, uint32_t n, uint64_t m, uint64_t seed, uint64_t *hist,
                              uint32_t nbins, double *kernel_ms) {
    clear_error();
    const uint64_t bounds[2] = {0, m};
    return an_mc_ranges(ctx, A, n, bounds, 1, seed, hist, nbins, kernel_ms);
}

extern "C" cr_status cr_an_mc_ranges(cr_context *ctx, uint64_t A, uint32_t n, const uint64_t *bounds,
                                     uint32_t count, uint64_t seed, uint64_t *hists, uint32_t nbins,
                                     double *kernel_ms) {
    clear_error();
    return an_mc_ranges(ctx, A, n, bounds, count, seed, hists, nbins, kernel_ms);
}
