// Extended-Hamming weight histograms of ranges of consecutive data words (gfx950):
// the counts ham_kernel would collect word by word (hamming.hip), from the
// structure of the code.
//
// The weight of data word d is popcount(d) + popcount(S(d)), S(d) its r parity
// bits, linear over GF(2).  A range is at most two blocks {d0 | x : x < 2^m} of
// each size (the masks and the data width wrap it modulo 2^k), and in a block
//   weight = popcount(d0) + popcount(x) + popcount(S(d0) ^ S(x)),
// so with J_m[j][s] = #{x < 2^m : popcount(x) = j, S(x) = s} a block adds J_m[j][s]
// to the weight popcount(d0) + j + popcount(S(d0) ^ s).  J_{m+1}[j][s] = J_m[j][s] +
// J_m[j - 1][s ^ S(2^m)]: k steps over (k + 1) * 2^r counters in LDS, whatever
// the number of words.
//
// One workgroup a range, bound by the barriers of its k steps and the LDS
// round trips between them; threads run along the parity values of one popcount,
// so neither the table nor the 64 histogram columns conflict.  Measured (39,32)
// code: a call for 2^20 aligned words 32 us, for 2^30 words at an odd place
// 43 us; word by word 39 and 541 us.
#include <algorithm>

#include "cr_device.h"
#include "cr_internal.h"

namespace cr {
namespace {

using namespace dev;

constexpr uint32_t kThreads = 512;
constexpr uint32_t kTable = 65 * 128;               // J[j * 2^r + s]: popcounts 0 .. 64, r <= 7 parity bits
constexpr uint32_t kPerThread = (kTable + kThreads - 1) / kThreads;
constexpr uint32_t kWeights = 72;                   // weights 0 .. 71
constexpr uint32_t kLane = 64;                      // histogram columns
constexpr size_t kLds = (kTable + kWeights * kLane) * sizeof(unsigned long long) + sizeof(HamRange);

__global__ __launch_bounds__(kThreads) void ham_range_kernel(const HamRange *__restrict__ jobs, const HamRange single,
                                                             const DirectResult direct) {
    extern __shared__ unsigned long long lds64[];
    unsigned long long *const J = lds64, *const hist = J + kTable;
    HamRange &job = *reinterpret_cast<HamRange *>(hist + kWeights * kLane);
    if (!jobs) direct_start(direct);
    const uint32_t tid = threadIdx.x;
    // the request in one round of loads: kernel arguments lie in host memory
    const unsigned long long *src = reinterpret_cast<const unsigned long long *>(jobs ? jobs + blockIdx.x : &single);
    for (uint32_t e = tid; e < sizeof(HamRange) / 8; e += kThreads) reinterpret_cast<unsigned long long *>(&job)[e] = src[e];
    for (uint32_t e = tid; e < kTable; e += kThreads) J[e] = e == 0;  // the empty word
    for (uint32_t e = tid; e < kWeights * kLane; e += kThreads) hist[e] = 0;
    __syncthreads();
    const uint32_t r = uniform32(job.r), nsyn = 1u << r, nblocks = uniform32(job.nblocks);
    uint32_t next = 0;
    for (uint32_t m = 0;; ++m) {
        for (; next < nblocks && uniform32(job.blocks[next].m) == m; ++next) {
            const HamRange::Block b = job.blocks[next];
            // consecutive threads: consecutive parity values of one popcount
            for (uint32_t e = tid; e < (m + 1) * nsyn; e += kThreads) {
                const uint32_t j = e >> r, s = e & (nsyn - 1);
                const unsigned long long n = J[e];
                if (n)
                    __hip_atomic_fetch_add(hist + (b.ones + j + __popc(s ^ b.parity)) * kLane + (s & (kLane - 1)),
                                           n * b.weight, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            }
        }
        if (next == nblocks) break;  // blocks are in order of m
        // J_{m+1}: popcount j from j and j - 1, parities shifted by those of 2^m
        const uint32_t col = uniform32(job.cols[m]), n = (m + 2) * nsyn;
        unsigned long long v[kPerThread];
#pragma unroll
        for (uint32_t u = 0; u < kPerThread; ++u) {
            if (u * kThreads >= n) break;
            const uint32_t e = tid + u * kThreads;
            v[u] = e >= nsyn && e < n ? J[(e - nsyn) ^ col] : 0;
        }
        __syncthreads();
#pragma unroll
        for (uint32_t u = 0; u < kPerThread; ++u) {
            if (u * kThreads >= n) break;
            if (v[u]) J[tid + u * kThreads] += v[u];
        }
        __syncthreads();
    }
    __syncthreads();
    const uint32_t lane = tid & 63;
    for (uint32_t w = tid / 64; w < job.nbins; w += kThreads / 64) {
        unsigned long long s = w < kWeights ? hist[w * kLane + lane] : 0;
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) s += __shfl_xor(s, d, 64);
        if (lane == 0) {
            if (jobs)
                job.out[w] = s;
            else
                direct.host[w] = s;
        }
    }
    if (!jobs && tid == 0) direct.host[kDirectBins + 1] = (unsigned long long)wall_clock64();
}

}  // namespace

// Blocks of [first, first + count) modulo 2^k, in order of size.
void ham_range_job(uint64_t first, uint64_t count, uint32_t k, const uint64_t masks[7], HamRange *job) {
    using u128 = unsigned __int128;
    job->nblocks = 0;
    const u128 size = (u128)1 << k;
    const uint64_t turns = k < 64 ? count >> k : 0;  // whole turns round the 2^k words
    const u128 n = (u128)count - ((u128)turns << k), a = k < 64 ? (u128)(first & ((1ull << k) - 1)) : (u128)first;
    auto parities = [&](uint64_t x) {
        uint32_t s = 0;
        for (int t = 0; t < 7; ++t) s |= (uint32_t)(__builtin_popcountll(x & masks[t]) & 1) << t;
        return s;
    };
    for (uint32_t m = 0; m < k; ++m) job->cols[m] = parities(1ull << m);
    auto block = [&](uint64_t d0, uint64_t weight, uint32_t m) {
        job->blocks[job->nblocks++] = {weight, (uint16_t)m, (uint16_t)__builtin_popcountll(d0),
                                       (uint16_t)parities(d0), 0};
    };
    auto add = [&](u128 lo, u128 hi) {
        for (uint32_t m = 0; lo < hi; ++m, lo >>= 1, hi >>= 1) {
            if (lo & 1) block((uint64_t)(lo++ << m), 1, m);
            if (lo < hi && (hi & 1)) block((uint64_t)(--hi << m), 1, m);
        }
    };
    if (a + n <= size) {
        add(a, a + n);
    } else {
        add(a, size);
        add(0, a + n - size);
    }
    if (turns) block(0, turns, k);
    std::stable_sort(job->blocks, job->blocks + job->nblocks,
                     [](const HamRange::Block &x, const HamRange::Block &y) { return x.m < y.m; });
}

cr_status launch_ham_ranges(const HamRange *d_jobs, uint32_t njobs, const HamRange *single,
                            const dev::DirectResult &out, hipStream_t stream) {
    const HamRange one = single ? *single : HamRange{};
    hipLaunchKernelGGL(ham_range_kernel, dim3(single ? 1 : njobs), dim3(kThreads), kLds, stream,
                       single ? (const HamRange *)nullptr : d_jobs, one, out);
    CR_HIP(hipGetLastError());
    return CR_OK;
}

}  // namespace cr
