// Device helpers shared by the histogram kernels (gfx950, wave64).
//
// All histogram kernels use the same LDS scheme: one single-wave workgroup
// owns rows of 64 uint32 counters, one row per distance/weight bin and one
// counter per lane (row stride 64 dwords), so every per-pair ds_add_u32 lands
// in the lane's own bank whatever the bin is.  Rows are flushed to 64-bit
// device histograms with one atomic per bin.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace cr {
namespace dev {

constexpr uint32_t kStride = 64;  // dwords between LDS histogram rows (one per lane)

// readfirstlane returns int: go through uint32_t so the low dword is not sign-extended
__device__ __forceinline__ uint32_t uniform32(uint32_t x) {
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)x);
}
__device__ __forceinline__ uint64_t uniform64(uint64_t x) {
    return ((uint64_t)uniform32((uint32_t)(x >> 32)) << 32) | (uint64_t)uniform32((uint32_t)x);
}

__device__ __forceinline__ void lds_inc(uint32_t *p) {
    __hip_atomic_fetch_add(p, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

__device__ __forceinline__ void lds_clear(uint32_t *lds, uint32_t rows) {
    for (uint32_t b = 0; b < rows; ++b) lds[b * kStride + threadIdx.x] = 0;
    __syncthreads();
}

// Adds every lane column of rows [first, nbins) to out[] and clears the rows.
// Lane l reduces row l (and l+64); at step s it reads column (s+l) mod 64, so
// the 64 lanes of one read hit 64 different banks.
__device__ inline void flush_rows(uint32_t *lds, uint32_t first, uint32_t nbins, unsigned long long *out) {
    __syncthreads();
    const uint32_t lane = threadIdx.x;
    for (uint32_t b = lane; b < nbins; b += 64) {
        uint32_t *row = lds + b * kStride;
        unsigned long long s = 0;
#pragma unroll 8
        for (uint32_t step = 0; step < 64; ++step) {
            const uint32_t l = (step + lane) & 63u;
            s += row[l];
            row[l] = 0;
        }
        if (s && b >= first) atomicAdd(out + b, s);
    }
    __syncthreads();
}

// Histogram copies: a histogram of nbins entries may be kept as `copies`
// copies (a power of two; 0 means 1), hist_copy_stride(nbins) entries apart,
// each on whole 128-byte lines; wave b flushes into copy b mod copies and the
// host sums the copies.  Many waves flushing one histogram otherwise queue
// their atomics on its few cache lines.
constexpr uint32_t kHistCopies = 32;
__host__ __device__ inline uint64_t hist_copy_stride(uint32_t nbins) { return ((uint64_t)nbins + 15) & ~15ull; }
__device__ __forceinline__ unsigned long long *hist_copy(unsigned long long *out, uint32_t nbins, uint32_t copies) {
    const uint32_t c = copies > 1 ? (blockIdx.x & (copies - 1)) : 0;
    return out + (uint64_t)c * hist_copy_stride(nbins);
}

// A call of one launch: the workgroups add to the histogram copies, the last
// one to finish sums them into pinned host memory.  The copies, the queue head
// and the tickets are zero between launches: the last workgroup leaves them so,
// so a call needs no fill before and no copy after its kernel (only one after
// a call that ended early does).
struct DirectResult {
    unsigned long long *copies = nullptr;  // kHistCopies copies, hist_copy_stride(nbins) apart
    unsigned long long *queue = nullptr;   // work-queue heads, kQueuePitch apart
    unsigned int *tickets = nullptr;       // workgroups that are done, by groups of them, then the groups
    unsigned long long *host = nullptr;    // nbins results; from kDirectBins: device clock at the start, at the end
};
constexpr uint32_t kDirectBins = 80;  // largest copy stride
// Device-scope atomics on one address serialize at about 12.5 ns, so the
// workgroups count themselves in groups, each on a cache line of its own.
constexpr uint32_t kTicketGroups = 64, kTicketPitch = 32;  // 32-bit tickets between two groups
// A launch of many short items divides them over kQueues heads for the same
// reason (most kernels use the first alone).
constexpr uint32_t kQueues = 8, kQueuePitch = 16;
constexpr size_t kDirectEntries =
    (size_t)kHistCopies * kDirectBins + kQueues * kQueuePitch + (kTicketGroups + 1) * kTicketPitch / 2;

// A result; system scope, so that it goes past the caches.
__device__ __forceinline__ void direct_store(const DirectResult &r, uint32_t i, unsigned long long x) {
    __hip_atomic_store(r.host + i, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The call's device time by the device's constant-rate clock: events around
// the launch cost 9 to 18 us of a 15 us call.
__device__ __forceinline__ void direct_start(const DirectResult &r) {
    if (blockIdx.x == 0 && threadIdx.x == 0) direct_store(r, kDirectBins, (unsigned long long)wall_clock64());
}

// Called by every thread of the workgroup that has written the results.  The
// end clock tells the host that they are there: it is written when every
// wave's stores have been acknowledged.
__device__ __forceinline__ void direct_end(const DirectResult &r) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) direct_store(r, kDirectBins + 1, (unsigned long long)wall_clock64());
}

// Called by every thread of every workgroup (a multiple of 64 threads) after
// its last addition; flag: one LDS dword.  The copies are only touched by
// device-scope atomics, which all XCDs see: waiting for them to complete before
// the ticket orders them, without the L2 write-back of a device-scope fence
// (measured at 55 us for 256 workgroups of 16 waves).
__device__ inline void direct_finish(const DirectResult &r, uint32_t nbins, uint32_t *flag) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) {
        const uint32_t g = blockIdx.x % kTicketGroups, groups = gridDim.x < kTicketGroups ? gridDim.x : kTicketGroups;
        const uint32_t members = (gridDim.x - g + kTicketGroups - 1) / kTicketGroups;
        bool last = __hip_atomic_fetch_add(r.tickets + (g + 1) * kTicketPitch, 1u, __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_AGENT) == members - 1;
        if (last)
            last = __hip_atomic_fetch_add(r.tickets, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == groups - 1;
        *flag = last;
    }
    __syncthreads();
    if (!*flag) return;
    // thread (b, c): copy c of distance b; eight exchanges in flight a thread
    const uint32_t c = threadIdx.x & (kHistCopies - 1), step = blockDim.x / kHistCopies;
    const uint64_t stride = hist_copy_stride(nbins);
    for (uint32_t b0 = threadIdx.x / kHistCopies; b0 < nbins; b0 += 8 * step) {
        unsigned long long s[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const uint32_t b = b0 + u * step;
            s[u] = b < nbins ? __hip_atomic_exchange(r.copies + c * stride + b, 0ull, __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_AGENT)
                             : 0;
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
#pragma unroll
            for (int d = kHistCopies / 2; d > 0; d >>= 1) s[u] += __shfl_xor(s[u], d, kHistCopies);
            if (c == 0 && b0 + u * step < nbins) direct_store(r, b0 + u * step, s[u]);
        }
    }
    for (uint32_t g = threadIdx.x; g <= kTicketGroups; g += blockDim.x)
        __hip_atomic_store(r.tickets + g * kTicketPitch, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (threadIdx.x < kQueues)
        __hip_atomic_store(r.queue + threadIdx.x * kQueuePitch, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    direct_end(r);
}

// Work-queue head: lane 0 takes the next item, every lane sees it.
__device__ __forceinline__ uint64_t next_item(unsigned long long *counter) {
    uint64_t t = 0;
    if (threadIdx.x == 0) t = atomicAdd(counter, 1ull);
    return uniform64(t);
}

// Item order of the persistent kernels (every launch has at most as many
// waves W = gridDim.x as items): wave b's first item is item b, taken without
// an atomic; its later items come from the work queue at `counter`, whose
// k-th step hands out item W + k, or, with counter == nullptr (a static
// assignment), are b + W, b + 2W, ...  Each queue step is a device-scope
// atomic on one address, serialized at about 12.5 ns on MI355X.
__device__ __forceinline__ uint64_t first_item() { return blockIdx.x; }
__device__ __forceinline__ uint64_t following_item(unsigned long long *counter, uint64_t t) {
    return counter ? (uint64_t)gridDim.x + next_item(counter) : t + gridDim.x;
}

// The same over n <= kQueues heads: item t belongs to the queue t mod n, wave w
// to the queue w mod n.  The launch has at least n waves, or as many as items
// (each then has one and none is left): a queue without a wave is never served.
__device__ __forceinline__ uint64_t following_item_of(unsigned long long *heads, uint32_t n) {
    const uint32_t q = blockIdx.x % n, waves = (gridDim.x - q + n - 1) / n;
    return q + (uint64_t)n * (waves + next_item(heads + q * kQueuePitch));
}

// Philox4x32-10 (Salmon, Moraes, Dror, Shaw, SC'11): ten rounds of the 4x32
// Philox S-box, multipliers 0xD2511F53 / 0xCD9E8D57, Weyl key increments
// 0x9E3779B9 / 0xBB67AE85.  c is the counter on input, the output on return.
// A round is two 32x32->64 products (v_mad_u64_u32) and two three-input XORs
// (v_bitop3_b32 with truth table 0x96, the key in a scalar register).
__device__ __forceinline__ void philox4x32_10(uint32_t (&c)[4], uint32_t k0, uint32_t k1) {
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        const uint64_t p0 = (uint64_t)0xD2511F53u * c[0];
        const uint64_t p1 = (uint64_t)0xCD9E8D57u * c[2];
        const uint32_t x0 = __builtin_amdgcn_bitop3_b32((uint32_t)(p1 >> 32), c[1], k0, 0x96);
        const uint32_t x2 = __builtin_amdgcn_bitop3_b32((uint32_t)(p0 >> 32), c[3], k1, 0x96);
        c[1] = (uint32_t)p1;
        c[3] = (uint32_t)p0;
        c[0] = x0;
        c[2] = x2;
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
    }
}

// Multipliers and round keys in vector registers.  v_bitop3, v_xor, v_and and the like with
// vector operands only issue for two waves of a SIMD at a time: 53 to 66e12 lane
// operations/s; with a scalar operand 37e12, as the multiplications do.  Blocks
// alone, 4 waves a SIMD: 0.78e12/s with scalar keys, 0.92e12/s with these.
struct PhiloxKeys {
    uint32_t a[10], b[10], m0, m1;
};
__device__ __forceinline__ uint32_t vector_copy(uint32_t s) {
    uint32_t v;
    asm("v_mov_b32 %0, %1" : "=v"(v) : "s"(s));
    return v;
}
__device__ __forceinline__ PhiloxKeys philox_keys(uint64_t seed) {
    PhiloxKeys k;
#pragma unroll
    for (uint32_t r = 0; r < 10; ++r) {
        k.a[r] = vector_copy((uint32_t)seed + r * 0x9E3779B9u);
        k.b[r] = vector_copy((uint32_t)(seed >> 32) + r * 0xBB67AE85u);
    }
    k.m0 = vector_copy(0xD2511F53u);
    k.m1 = vector_copy(0xCD9E8D57u);
    return k;
}
// Rounds FIRST .. 9 of philox4x32_10.
template <int FIRST>
__device__ __forceinline__ void philox_rounds(uint32_t (&c)[4], const PhiloxKeys &k) {
#pragma unroll
    for (int r = FIRST; r < 10; ++r) {
        const uint64_t p0 = (uint64_t)k.m0 * c[0];
        const uint64_t p1 = (uint64_t)k.m1 * c[2];
        c[0] = __builtin_amdgcn_bitop3_b32((uint32_t)(p1 >> 32), c[1], k.a[r], 0x96);
        c[2] = __builtin_amdgcn_bitop3_b32((uint32_t)(p0 >> 32), c[3], k.b[r], 0x96);
        c[1] = (uint32_t)p1;
        c[3] = (uint32_t)p0;
    }
}

// Tag in the fourth counter word of the library's Monte Carlo streams.
constexpr uint32_t kMcTag = 0x43520001u;

}  // namespace dev
}  // namespace cr
