// Pair-distance histograms of short codes in one launch (gfx950): the same
// raw[] as the pair kernel for fewer than 2^16 words, where a call is bound by
// its launches, copies and tail as much as by its pairs.
//
// Rows in blocks of 64 * R (R codewords a lane in registers), the columns from
// the block's first row to the end in steps of one wave-uniform column; the
// steps of all blocks in a row are dealt to the waves in equal shares, so every
// wave does the same work.  All waves of a workgroup count into one LDS
// histogram (a counter a distance and lane, ds_add_u32 to the lane's own bank);
// the last workgroup to finish writes the sums to pinned host memory
// (direct_finish).  A call of 2^8 words takes one workgroup.  Measured a call
// (device time): 2^8 words 13.5 us (3.5), 2^13 20 us (12); 10001 words 25 us,
// 20001 50 us, 50001 200 us; the pair kernel with its fill, job upload, result
// copy and timing events 43 us (15), 49 us (20), 48, 73 and 344 us.  At 2^16 words
// both take 0.32 ms (one workgroup a CU here).
#include <algorithm>

#include "cr_device.h"
#include "cr_internal.h"

namespace cr {
namespace {

using namespace dev;

constexpr uint32_t kThreads = 1024;
constexpr uint32_t kWaves = kThreads / 64;
constexpr uint32_t kRows = 67;  // distances 0 .. 64 and the row of masked pairs

struct ShortJob {
    uint64_t A;
    uint32_t N, R, steps, share;  // words, rows a lane, column steps of all blocks, steps of a wave
    uint32_t nbins;
};

// Columns [j0, j1) against row block b.
template <int R, bool W2>
__device__ __forceinline__ void columns(uint32_t *lane_col, uint64_t A, uint32_t row0, uint32_t j0, uint32_t j1) {
    const uint32_t lane = threadIdx.x & 63;
    uint32_t lo[R], hi[R], row[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        row[r] = row0 + r * 64 + lane;
        const uint64_t w = A * row[r];
        lo[r] = (uint32_t)w;
        hi[r] = (uint32_t)(w >> 32);
    }
    uint64_t v = uniform64(A * j0);
    uint32_t j = j0;
    // up to the block's last row a column meets only the rows before it
    for (const uint32_t diag = min(j1, row0 + 64 * R); j < diag; ++j, v += A)
#pragma unroll
        for (int r = 0; r < R; ++r) {
            uint32_t d = __popc(lo[r] ^ (uint32_t)v);
            if (W2) d += __popc(hi[r] ^ (uint32_t)(v >> 32));
            lds_inc(lane_col + (j > row[r] ? d : kRows - 1) * kStride);
        }
#pragma unroll 4
    for (; j < j1; ++j, v += A)
#pragma unroll
        for (int r = 0; r < R; ++r) {
            uint32_t d = __popc(lo[r] ^ (uint32_t)v);
            if (W2) d += __popc(hi[r] ^ (uint32_t)(v >> 32));
            lds_inc(lane_col + d * kStride);
        }
}

template <int R, bool W2>
__global__ __launch_bounds__(kThreads) void short_kernel(ShortJob job, DirectResult out) {
    __shared__ uint32_t lds[kRows * kStride];
    __shared__ uint32_t flag;
    direct_start(out);
    for (uint32_t i = threadIdx.x; i < kRows * kStride; i += kThreads) lds[i] = 0;
    __syncthreads();
    const uint32_t wave = uniform32(threadIdx.x / 64), lane = threadIdx.x & 63;
    constexpr uint32_t RB = 64 * R;
    // this wave's steps [s, end) of the blocks' columns one after the other
    uint32_t s = (blockIdx.x * kWaves + wave) * job.share;
    const uint32_t end = min(s + job.share, job.steps);
    uint32_t first = 0;  // row block and the steps before it
    uint32_t before = 0;
    while (s < end) {
        while (s - before >= job.N - first) {
            before += job.N - first;
            first += RB;
        }
        const uint32_t j0 = first + (s - before), n = min(end - s, job.N - j0);
        columns<R, W2>(lds + lane, job.A, first, j0, j0 + n);
        s += n;
    }
    __syncthreads();
    // a wave sums a row: its 64 lanes' counters
    for (uint32_t b = wave; b < job.nbins; b += kWaves) {
        uint32_t x = lds[b * kStride + lane];
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) x += __shfl_xor(x, d, 64);
        if (lane == 0) {
            if (gridDim.x == 1)
                direct_store(out, b, x);
            else if (x)
                atomicAdd(hist_copy(out.copies, job.nbins, kHistCopies) + b, (unsigned long long)x);
        }
    }
    if (gridDim.x > 1)
        direct_finish(out, job.nbins, &flag);
    else
        direct_end(out);
}

const void *short_kernel_for(uint32_t R, bool w2) {
    if (R == 1) return w2 ? reinterpret_cast<const void *>(&short_kernel<1, true>)
                          : reinterpret_cast<const void *>(&short_kernel<1, false>);
    return w2 ? reinterpret_cast<const void *>(&short_kernel<4, true>)
              : reinterpret_cast<const void *>(&short_kernel<4, false>);
}

}  // namespace

cr_status launch_short_pairs(uint64_t A, uint32_t N, uint32_t nbins, const dev::DirectResult &out, int cus,
                             hipStream_t stream) {
    if (N == 0 || N > kShortWords || nbins > kRows - 1)
        return fail(CR_ERR_INVALID_ARGUMENT, "short pairs: %u words, %u distances", N, nbins);
    ShortJob job{};
    job.A = A;
    job.N = N;
    job.R = N >= 2048 ? 4 : 1;
    job.nbins = nbins;
    for (uint32_t b = 0; b < N; b += 64 * job.R) job.steps += N - b;
    // at least 32 steps a wave; a counter is below 2^16 * R
    const uint32_t groups = std::min<uint32_t>((uint32_t)cus, std::max<uint32_t>(1, job.steps / (32 * kWaves)));
    job.share = (job.steps + groups * kWaves - 1) / (groups * kWaves);
    dev::DirectResult a_out = out;
    void *args[] = {&job, &a_out};
    CR_HIP(hipLaunchKernel(short_kernel_for(job.R, (unsigned __int128)A * (N - 1) >> 32 != 0), dim3(groups),
                           dim3(kThreads), args, 0, stream));
    return CR_OK;
}

}  // namespace cr
