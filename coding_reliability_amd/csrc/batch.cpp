// Batched exhaustive AN histograms: many codes, one persistent launch,
// optionally replayed from a captured hipGraph; plus the autotuner.
#include <algorithm>
#include <chrono>
#include <cstring>
#include <numeric>
#include <vector>

#include "cr_device.h"
#include "cr_internal.h"

namespace cr {

namespace {

struct BatchLayout {
    std::vector<PairJob> jobs;      // codes of the pair kernel, longest first
    PairLaunchConfig cfg;
    uint64_t total_items = 0;
    std::vector<SlicedJob> sliced;  // codes of the sliced kernel, longest first
    uint64_t sliced_items = 0;
    size_t job_bytes() const { return sliced.size() * sizeof(SlicedJob) + jobs.size() * sizeof(PairJob); }
    // device layout: the sliced jobs, then the pair jobs
    hipError_t upload(void *d, hipStream_t stream) const {
        const size_t n = sliced.size() * sizeof(SlicedJob);
        hipError_t e = n ? hipMemcpyAsync(d, sliced.data(), n, hipMemcpyHostToDevice, stream) : hipSuccess;
        if (e == hipSuccess && !jobs.empty())
            e = hipMemcpyAsync(static_cast<char *>(d) + n, jobs.data(), jobs.size() * sizeof(PairJob),
                               hipMemcpyHostToDevice, stream);
        return e;
    }
};
static_assert(alignof(PairJob) == alignof(SlicedJob) && sizeof(SlicedJob) % alignof(PairJob) == 0, "job array layout");

// Builds the work lists, jobs sorted by pair count (longest first), each
// writing to d_hist + c*stride: codes of 2^k words from k = 11 on go to the
// sliced kernel, the others to the pair kernel with the chunk width chosen so
// that items carry about total_pairs/(items_per_wave * resident waves) pairs.
cr_status build_batch(cr_context *ctx, const cr_an_code *codes, uint32_t ncodes, uint32_t stride,
                      const cr_pair_tuning *tuning, unsigned long long *d_hist, BatchLayout &L) {
    if (!codes || ncodes == 0) return fail(CR_ERR_INVALID_ARGUMENT, "empty batch");
    const uint32_t ipw = tuning && tuning->items_per_wave ? tuning->items_per_wave : 16;
    uint32_t max_need = 0;  // of the pair kernel's codes: its waves per CU follow from their bins
    long double total_pairs = 0, short_pairs = 0, sliced_pairs = 0;
    uint64_t most_words = 0, most_sliced = 0;
    L.jobs.reserve(ncodes);
    std::vector<uint32_t> sliced;  // codes that the sliced kernel can take
    auto to_pairs = [&](uint32_t c) {
        PairJob j{};
        j.A = codes[c].A;
        j.N = codes[c].num_words;
        j.out = d_hist + (size_t)c * stride;
        j.nbins = pair_max_distance(j.A, j.N) + 1;
        j.mode = pair_mode(j.A, j.N);
        L.cfg.wide = L.cfg.wide || j.mode == kModeWide;
        L.jobs.push_back(j);
        max_need = std::max(max_need, j.nbins);
        const long double pairs = (long double)j.N * (long double)(j.N - 1) / 2;
        total_pairs += pairs;
        if (j.N < (1ull << 15)) short_pairs += pairs;
        most_words = std::max(most_words, j.N);
    };
    for (uint32_t c = 0; c < ncodes; ++c) {
        const uint64_t A = codes[c].A, N = codes[c].num_words;
        if (A == 0 || N == 0) return fail(CR_ERR_INVALID_ARGUMENT, "code %u: A and num_words must be >= 1", c);
        if ((unsigned __int128)(N - 1) * A >> 64) return fail(CR_ERR_UNSUPPORTED, "code %u exceeds 64-bit codewords", c);
        const uint32_t need = pair_max_distance(A, N) + 1;
        if (need > stride) return fail(CR_ERR_INVALID_ARGUMENT, "code %u needs %u bins > stride %u", c, need, stride);
        SlicedJob sj;
        if (sliced_job(A, N, &sj)) {
            sj.out = d_hist + (size_t)c * stride;
            sj.nbins = need;
            L.sliced.push_back(sj);
            sliced.push_back(c);
            sliced_pairs += (long double)N * (long double)N / 2;
            most_sliced = std::max(most_sliced, N);
        } else {
            to_pairs(c);
        }
    }
    // as for single codes: short codes waste less of a row block of 128 words
    // than of one of 512 (16384 codes of 2^8 words 0.48 ms with 8 rows a lane, 0.20
    // with 2; 4096 codes of 2^10 words 0.64 and 0.46)
    const uint32_t R = tuning && tuning->rows_per_lane ? tuning->rows_per_lane : 2 * short_pairs >= total_pairs ? 2 : 8;
    // Few pairs of the sliced kernel's codes do not pay for its launch (14 us at
    // least): they go with the pair kernel's codes where those take a wave as long,
    // a row block of 64 R words against itself (31 us with 4 rows a lane, 86 with
    // 8), are not too long for so few rows, and need no matrix instructions (whose
    // kernel is the slower one for other codes).  60 codes of 3000 words and four of
    // 2^11 102 -> 88 us (4 rows 110 -> 94, 8 rows 172 -> 156); not so 60 of 200 words
    // and one of 2^13 57 -> 69 (8 rows 82 -> 112).
    if (!L.jobs.empty() && !L.cfg.wide && sliced_pairs < 2.5e7L * std::max(R, 4u) && most_words > 48ull * R &&
        most_sliced <= 2048ull * R) {
        for (uint32_t c : sliced) to_pairs(c);
        L.sliced.clear();
    }
    L.cfg.R = R;
    L.cfg.lds_rows = std::max(max_need, 1u) + 1;
    L.cfg.waves = tuning ? tuning->waves : 0;
    L.cfg.zero_counter = false;
    const uint32_t per_cu = pair_waves_per_cu(R, L.cfg.lds_rows, L.cfg.wide);
    if (per_cu == 0) return fail(CR_ERR_INVALID_ARGUMENT, "rows_per_lane must be 2, 4, 8 or 16 (got %u)", R);
    const long double waves = (long double)per_cu * ctx->cus;
    const long double target = std::max<long double>(total_pairs / (ipw * waves), 1.0L);
    const uint64_t RB = 64ull * R;
    const uint64_t qmax = std::max<uint64_t>(((1ull << 30) / R) / RB, 1);
    for (PairJob &j : L.jobs) {
        uint64_t Q = (uint64_t)(target / ((long double)RB * RB));
        Q = std::min<uint64_t>(std::max<uint64_t>(Q, 1), qmax);
        pair_job_geometry(j, R, (uint32_t)Q);
    }
    std::stable_sort(L.jobs.begin(), L.jobs.end(), [](const PairJob &a, const PairJob &b) {
        return (unsigned __int128)a.N * a.N > (unsigned __int128)b.N * b.N;
    });
    uint64_t total = 0;
    for (auto &j : L.jobs) {
        j.item_begin = total;
        total += j.items;
    }
    L.total_items = total;
    // a head hands out an item in 12.5 ns, in which the device counts 2^17
    // pairs: 16384 codes of 2^4 words 0.22 -> 0.06 ms with eight heads
    L.cfg.heads = total_pairs < (long double)total * (1 << 17) ? dev::kQueues : 1;
    std::stable_sort(L.sliced.begin(), L.sliced.end(),
                     [](const SlicedJob &a, const SlicedJob &b) { return a.k > b.k; });
    sliced_ranges(L.sliced, ctx->cus, &L.sliced_items);
    return CR_OK;
}

// The work-queue heads lie behind the n counts of the histograms, on lines of
// their own, so that one fill clears both: the pair kernel's, then the sliced one's.
constexpr size_t kCounters = dev::kQueues * dev::kQueuePitch + 1;
size_t counters_at(size_t n) { return (n + dev::kQueuePitch - 1) / dev::kQueuePitch * dev::kQueuePitch; }
size_t batch_entries(size_t n) { return counters_at(n) + kCounters; }

// Both launches, the heads cleared.
cr_status launch_batch(cr_context *ctx, const BatchLayout &L, void *d_jobs, unsigned long long *counters) {
    const SlicedJob *sliced = static_cast<const SlicedJob *>(d_jobs);
    if (!L.sliced.empty())
        CR_TRY(launch_sliced(sliced, (uint32_t)L.sliced.size(), L.sliced_items, counters + kCounters - 1, ctx->cus,
                             ctx->stream));
    if (!L.jobs.empty())
        CR_TRY(launch_pairs(reinterpret_cast<const PairJob *>(sliced + L.sliced.size()), (uint32_t)L.jobs.size(),
                            L.total_items, counters, L.cfg, ctx->cus, ctx->stream, nullptr, nullptr));
    return CR_OK;
}

}  // namespace

}  // namespace cr

using namespace cr;

struct cr_batch_plan {
    cr_context *ctx = nullptr;
    uint32_t ncodes = 0, stride = 0;
    DeviceBuffer jobs, hist;
    HostBuffer host;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
};

extern "C" {

cr_status cr_an_batch(cr_context *ctx, const cr_an_code *codes, uint32_t ncodes, uint64_t *raw, uint32_t stride,
                      const cr_pair_tuning *tuning, double *kernel_ms) {
    clear_error();
    if (!ctx || !raw) return fail(CR_ERR_INVALID_ARGUMENT, "NULL argument");
    CR_HIP(hipSetDevice(ctx->device));
    const size_t n = (size_t)ncodes * stride;
    CR_TRY(ctx->hist.reserve(batch_entries(n) * sizeof(uint64_t)));
    unsigned long long *const hist = ctx->hist.as<unsigned long long>();
    BatchLayout L;
    CR_TRY(build_batch(ctx, codes, ncodes, stride, tuning, hist, L));
    CR_TRY(ctx->jobs.reserve(L.job_bytes()));
    CR_TRY(fill_zero_u64(hist, batch_entries(n), ctx->stream));
    CR_HIP(L.upload(ctx->jobs.ptr, ctx->stream));
    if (kernel_ms) CR_HIP(hipEventRecord(ctx->ev0, ctx->stream));
    CR_TRY(launch_batch(ctx, L, ctx->jobs.ptr, hist + counters_at(n)));
    if (kernel_ms) CR_HIP(hipEventRecord(ctx->ev1, ctx->stream));
    CR_TRY(ctx->host.reserve(n * sizeof(uint64_t)));
    CR_HIP(hipMemcpyAsync(ctx->host.ptr, ctx->hist.ptr, n * sizeof(uint64_t), hipMemcpyDeviceToHost, ctx->stream));
    CR_HIP(hipStreamSynchronize(ctx->stream));
    memcpy(raw, ctx->host.ptr, n * sizeof(uint64_t));
    if (kernel_ms) {
        float ms = 0;
        CR_HIP(hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1));
        *kernel_ms = ms;
    }
    return CR_OK;
}

cr_status cr_batch_plan_destroy(cr_batch_plan *p) {
    if (!p) return CR_OK;
    if (p->ctx) (void)hipSetDevice(p->ctx->device);
    if (p->exec) (void)hipGraphExecDestroy(p->exec);
    if (p->graph) (void)hipGraphDestroy(p->graph);
    p->jobs.release();
    p->hist.release();
    p->host.release();
    delete p;
    return CR_OK;
}

cr_status cr_batch_plan_create(cr_context *ctx, const cr_an_code *codes, uint32_t ncodes, uint32_t stride,
                               const cr_pair_tuning *tuning, cr_batch_plan **out) {
    clear_error();
    if (!ctx || !out) return fail(CR_ERR_INVALID_ARGUMENT, "NULL argument");
    *out = nullptr;
    CR_HIP(hipSetDevice(ctx->device));
    cr_batch_plan *p = new cr_batch_plan();
    p->ctx = ctx;
    p->ncodes = ncodes;
    p->stride = stride;
    auto bail = [&](cr_status s) {
        cr_batch_plan_destroy(p);
        return s;
    };
    const size_t n = (size_t)ncodes * stride;
    cr_status s;
    if ((s = p->hist.reserve(batch_entries(n) * sizeof(uint64_t))) != CR_OK) return bail(s);
    unsigned long long *const hist = p->hist.as<unsigned long long>();
    if ((s = p->host.reserve(n * sizeof(uint64_t))) != CR_OK) return bail(s);
    BatchLayout L;
    if ((s = build_batch(ctx, codes, ncodes, stride, tuning, hist, L)) != CR_OK)
        return bail(s);
    if ((s = p->jobs.reserve(L.job_bytes())) != CR_OK) return bail(s);
    hipError_t e = L.upload(p->jobs.ptr, ctx->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);  // L goes with this call
    if (e != hipSuccess) return bail(fail(CR_ERR_DEVICE, "job upload failed: %s", hipGetErrorString(e)));
    // capture: zero histograms and queue heads, kernels, copy back
    e = hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal);
    if (e != hipSuccess) return bail(fail(CR_ERR_DEVICE, "graph capture failed: %s", hipGetErrorString(e)));
    cr_status cs = fill_zero_u64(hist, batch_entries(n), ctx->stream);
    if (cs == CR_OK) cs = launch_batch(ctx, L, p->jobs.ptr, hist + counters_at(n));
    if (cs == CR_OK) {
        e = hipMemcpyAsync(p->host.ptr, p->hist.ptr, n * sizeof(uint64_t), hipMemcpyDeviceToHost, ctx->stream);
        if (e != hipSuccess) cs = fail(CR_ERR_DEVICE, "capture of copy-back failed: %s", hipGetErrorString(e));
    }
    hipGraph_t g = nullptr;
    e = hipStreamEndCapture(ctx->stream, &g);
    p->graph = g;
    if (cs != CR_OK) return bail(cs);
    if (e != hipSuccess) return bail(fail(CR_ERR_DEVICE, "graph capture failed: %s", hipGetErrorString(e)));
    e = hipGraphInstantiate(&p->exec, p->graph, nullptr, nullptr, 0);
    if (e != hipSuccess) return bail(fail(CR_ERR_DEVICE, "graph instantiation failed: %s", hipGetErrorString(e)));
    *out = p;
    return CR_OK;
}

cr_status cr_batch_plan_run(cr_batch_plan *p, uint64_t *raw, double *elapsed_ms) {
    clear_error();
    if (!p) return fail(CR_ERR_INVALID_ARGUMENT, "NULL plan");
    cr_context *ctx = p->ctx;
    CR_HIP(hipSetDevice(ctx->device));
    CR_HIP(hipEventRecord(ctx->ev0, ctx->stream));
    CR_HIP(hipGraphLaunch(p->exec, ctx->stream));
    CR_HIP(hipEventRecord(ctx->ev1, ctx->stream));
    CR_HIP(hipStreamSynchronize(ctx->stream));
    if (raw) memcpy(raw, p->host.ptr, (size_t)p->ncodes * p->stride * sizeof(uint64_t));
    if (elapsed_ms) {
        float ms = 0;
        CR_HIP(hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1));
        *elapsed_ms = ms;
    }
    return CR_OK;
}

cr_status cr_autotune_batch(cr_context *ctx, const cr_an_code *codes, uint32_t ncodes, uint32_t repeats,
                            cr_pair_tuning *best, double *best_ms) {
    clear_error();
    if (!ctx || !best) return fail(CR_ERR_INVALID_ARGUMENT, "NULL argument");
    if (repeats == 0) repeats = 1;
    uint32_t stride = 0;
    for (uint32_t c = 0; c < ncodes; ++c) {
        if (codes[c].A == 0 || codes[c].num_words == 0) return fail(CR_ERR_INVALID_ARGUMENT, "bad code %u", c);
        stride = std::max(stride, pair_max_distance(codes[c].A, codes[c].num_words) + 1);
    }
    const uint32_t Rs[] = {4, 8, 16};
    const uint32_t ipws[] = {4, 16, 64};
    double bms = 1e300;
    cr_pair_tuning bt{};
    for (uint32_t R : Rs)
        for (uint32_t ipw : ipws) {
            cr_pair_tuning t{R, 0, 0, ipw};
            cr_batch_plan *p = nullptr;
            CR_TRY(cr_batch_plan_create(ctx, codes, ncodes, stride, &t, &p));
            double m = 1e300;
            for (uint32_t r = 0; r <= repeats; ++r) {  // first run warms up
                double ms = 0;
                cr_status s = cr_batch_plan_run(p, nullptr, &ms);
                if (s != CR_OK) {
                    cr_batch_plan_destroy(p);
                    return s;
                }
                if (r) m = std::min(m, ms);
            }
            cr_batch_plan_destroy(p);
            if (m < bms) {
                bms = m;
                bt = t;
            }
        }
    *best = bt;
    if (best_ms) *best_ms = bms;
    return CR_OK;
}

}  // extern "C"
