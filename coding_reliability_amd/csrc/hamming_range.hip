// Extended-Hamming weight histograms of ranges of consecutive data words (gfx950):
// the counts ham_kernel would collect word by word (hamming.hip), from the
// structure of the code.
//
// The weight of data word d is popcount(d) + popcount(S(d)), S(d) its r parity
// bits, linear over GF(2).  L_m[j][s] counts words by the popcount j and the
// parity bits s of their upper m bits; a further bit, of parity column c, gives
// L_{m+1}[j][s] = L_m[j][s] + L_m[j - 1][s ^ c].  The words below a bound v enter
// where they first differ from it: at each 1 bit of v the word with v's bits
// above it and a 0 there.  A range is the words below its end less those below
// its start (modulo 2^64, and with a count of all words where it passes 2^k: the
// masks and the data width wrap it), so one recursion with +1 and -1 entries
// gives its counts: k steps over at most (k + 1) * 2^r counters in LDS, whatever the
// number of words.
//
// One workgroup a range, two bits a step (four reads, a write), two tables in
// turn, so that a step is one barrier; bound by that latency (0.35 us a step of
// the (39,32) code, k = 64 by the LDS too).  Several counters of a thread in
// flight did not help, 512 threads took 24 us where 1024 take 23.  Measured, a call
// for 2^30 words of the (39,32) code 20 us (word by word 541 us), k = 64 42 us (a
// few words 33 us word by word, so they do not come here: hamming_api.cpp).
#include <algorithm>

#include "cr_device.h"
#include "cr_internal.h"

namespace cr {
namespace {

using namespace dev;

constexpr uint32_t kThreads = 1024;
constexpr uint32_t kWeights = 72;  // weights 0 .. 71
constexpr uint32_t kLane = 64;     // histogram columns

// Entries of one table: two rows of zeros, popcounts 0 .. k; at least the
// histogram, which takes the place of the table not in use at the end.
uint32_t table_entries(uint32_t k, uint32_t r) { return std::max((k + 3) << r, kWeights * kLane); }

__global__ __launch_bounds__(kThreads) void ham_range_kernel(const HamRange *__restrict__ jobs, const HamRange single,
                                                             uint32_t entries, const DirectResult direct) {
    extern __shared__ unsigned long long lds64[];
    if (!jobs) direct_start(direct);
    HamRange &job = *reinterpret_cast<HamRange *>(lds64 + 2 * entries);
    const uint32_t tid = threadIdx.x;
    // the request in one round of loads: kernel arguments lie in host memory
    const unsigned long long *src = reinterpret_cast<const unsigned long long *>(jobs ? jobs + blockIdx.x : &single);
    for (uint32_t e = tid; e < sizeof(HamRange) / 8; e += kThreads) reinterpret_cast<unsigned long long *>(&job)[e] = src[e];
    for (uint32_t e = tid; e < 2 * entries; e += kThreads) lds64[e] = 0;
    __syncthreads();
    const uint32_t r = uniform32(job.r), row = 1u << r, steps = uniform32(job.steps);
    uint32_t m = uniform32(job.start_bits);
    unsigned long long *from = lds64 + 2 * row, *to = from + entries;
    if (tid == 0)
        for (uint32_t i = 0; i < 4; ++i) from[job.start[i].at] += job.start[i].weight;
    __syncthreads();
    const uint32_t lane = tid & 63, wave = uniform32(tid / 64);
    // a step's numbers are read a step ahead; lane i < 6 of each wave holds entry i
    const uint32_t *next = reinterpret_cast<const uint32_t *>(job.step);
    const uint32_t mine = 1 + (lane < 6 ? lane : 5);
    uint32_t cols = next[0], enter = next[mine];
    for (uint32_t t = 0; t < steps; ++t, m += 2) {
        const uint32_t c1 = uniform32(cols & 0xFFFF), c2 = uniform32(cols >> 16), n = (m + 3) * row;
        const uint32_t at = enter & 0xFFFF;
        const long long sign = lane < 6 ? (int16_t)(enter >> 16) : 0;
        next += sizeof(HamRange::Step) / 4;
        if (t + 1 < steps) cols = next[0], enter = next[mine];
        for (uint32_t e = tid; e < n; e += kThreads)
            to[e] = from[e] + from[(int)(e ^ c1) - (int)row] + from[(int)(e ^ c2) - (int)row] +
                    from[(int)(e ^ c1 ^ c2) - 2 * (int)row];
        // by the wave that wrote the counter: a wave's LDS operations keep their order
        if (sign && (at % kThreads) / 64 == wave)
            __hip_atomic_fetch_add(to + at, (unsigned long long)sign, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        __syncthreads();
        unsigned long long *swap = from;
        from = to;
        to = swap;
    }
    // weights: consecutive threads take consecutive parity values of one popcount
    unsigned long long *const hist = to - 2 * row;
    for (uint32_t e = tid; e < kWeights * kLane; e += kThreads) hist[e] = 0;
    __syncthreads();
    for (uint32_t e = tid; e < (m + 1) * row; e += kThreads) {
        const unsigned long long n = from[e];
        const uint32_t s = e & (row - 1);
        if (n)
            __hip_atomic_fetch_add(hist + ((e >> r) + __popc(s)) * kLane + (s & (kLane - 1)), n, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    __syncthreads();
    for (uint32_t w = wave; w < job.nbins; w += kThreads / 64) {
        unsigned long long s = w < kWeights ? hist[w * kLane + lane] : 0;
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) s += __shfl_xor(s, d, 64);
        if (lane == 0) {
            if (jobs)
                job.out[w] = s;
            else
                direct_store(direct, w, s);
        }
    }
    if (!jobs) direct_end(direct);
}

}  // namespace

void ham_range_job(uint64_t first, uint64_t count, uint32_t k, const uint64_t masks[7], HamRange *job) {
    using u128 = unsigned __int128;
    const u128 size = (u128)1 << k;
    const uint64_t turns = k < 64 ? count >> k : 0;  // whole turns round the 2^k words
    const u128 n = (u128)count - ((u128)turns << k), a = (u128)first & (size - 1), b = a + n;
    // [a, b) = all words, turns + (b >= size) times, and those below b mod size, less those below a
    const uint64_t all = turns + (b >= size), bound[2] = {(uint64_t)a, (uint64_t)(b & (size - 1))};
    auto parities = [&](uint64_t x) {
        uint32_t s = 0;
        for (int t = 0; t < 7; ++t) s |= (uint32_t)(__builtin_popcountll(x & masks[t]) & 1) << t;
        return s;
    };
    const uint32_t r = job->r;
    auto at = [&](uint64_t x) { return ((uint32_t)__builtin_popcountll(x) << r) + parities(x); };
    // the word below bound i that leaves it at bit t, 0 if there is none
    auto leaves = [&](int i, uint32_t t, uint64_t *x) {
        if (!(bound[i] >> t & 1)) return false;
        *x = bound[i] & ~((2ull << t) - 1);
        return true;
    };
    uint64_t x = 0;
    // an odd width's top bit, or nothing, before the steps of two
    job->start_bits = k & 1;
    job->start[0] = {all, 0, 0};
    if (k & 1) {
        job->start[1] = {all, at(1ull << (k - 1)), 0};
        for (int i = 0; i < 2; ++i)
            if (leaves(i, k - 1, &x)) job->start[2 + i] = {i ? 1ull : ~0ull, at(x), 0};
    }
    job->steps = k / 2;
    for (uint32_t t = 0; t < k / 2; ++t) {
        const uint32_t hi = k - (k & 1) - 1 - 2 * t, lo = hi - 1;
        HamRange::Step &s = job->step[t];
        s.col[0] = (uint16_t)parities(1ull << hi);
        s.col[1] = (uint16_t)parities(1ull << lo);
        for (int i = 0; i < 2; ++i) {
            const int16_t sign = i ? 1 : -1;
            if (leaves(i, hi, &x)) {
                s.enter[3 * i] = {(uint16_t)at(x), sign};
                s.enter[3 * i + 1] = {(uint16_t)at(x | 1ull << lo), sign};
            }
            if (leaves(i, lo, &x)) s.enter[3 * i + 2] = {(uint16_t)at(x), sign};
        }
    }
}

cr_status launch_ham_ranges(const HamRange *d_jobs, uint32_t njobs, const HamRange *single, uint32_t max_k,
                            uint32_t max_r, const dev::DirectResult &out, hipStream_t stream) {
    const HamRange one = single ? *single : HamRange{};
    const uint32_t entries = table_entries(max_k, max_r);
    hipLaunchKernelGGL(ham_range_kernel, dim3(single ? 1 : njobs), dim3(kThreads),
                       2 * entries * sizeof(unsigned long long) + sizeof(HamRange), stream,
                       single ? (const HamRange *)nullptr : d_jobs, one, entries, out);
    CR_HIP(hipGetLastError());
    return CR_OK;
}

}  // namespace cr
