// Exhaustive pair-distance histogram kernel for AN codes (gfx950).
//
// Computes raw[b] = #{i<j : popcount(A*i ^ A*j) == b}, the quantity the
// reference kernel dancoding_shared accumulates
// (distance_distribution/src/an_coding.cu:50-105), with a different execution
// scheme:
//   * one wave per workgroup, persistent, pulling items from a global queue;
//   * R row codewords per lane live in VGPRs (A*i computed, never loaded);
//   * the column codeword is wave-uniform and advances in SGPRs (v += A), so a
//     pair costs one v_xor + one v_bcnt (+ bcnt accumulate of the constant
//     high-dword distance for 33..64-bit words) + one LDS address mad + one
//     ds_add_u32 into the lane's private column of the histogram (multipliers
//     above 2^22: the matrix cores compute the address, see pairs_wide);
//   * LDS histogram rows are 64 dwords (one per lane), so the bank of every
//     per-pair atomic is fixed by the lane whatever the distance is: the hot
//     loop never bank-conflicts; the flush reads each row in a lane-rotated
//     order, which is conflict free too; counters are flushed to the 64-bit
//     device histogram with one atomic per bin per flush, before any 32-bit
//     lane counter can wrap.
#include <atomic>

#include "cr_device.h"
#include "cr_internal.h"

namespace cr {

namespace {

using namespace dev;
constexpr uint32_t kUnroll = 4;  // columns per unrolled step

template <int R>
struct Rows {
    uint64_t w[R];  // codeword A*i_r
    uint64_t i[R];  // row index i_r
};

// Diagonal block: columns [j0, j1) are below (b+1)*RB, pairs with j <= i go to
// the dummy row.  Generic 64-bit path; at most RB columns per row block.
template <int R>
__device__ void pairs_masked(uint32_t *lane_col, const Rows<R> &rw, uint64_t A, uint64_t j0, uint64_t j1,
                             uint32_t dummy) {
    uint64_t v = A * j0;
    if constexpr (R == 16) {
        // XORs, then counts, then increments: left to itself the compiler may put
        // one pair behind the other (which it does depends on the rest of the
        // kernel), and a single wave, as of a short code, takes 15 % longer
        for (uint64_t j = j0; j < j1; ++j, v += A) {
            uint64_t x[R];
            uint32_t c[R];
#pragma unroll
            for (int r = 0; r < R; ++r) x[r] = rw.w[r] ^ v;
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int r = 0; r < R; ++r) c[r] = (uint32_t)__popcll(x[r]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int r = 0; r < R; ++r) lds_inc(lane_col + (j > rw.i[r] ? c[r] : dummy) * kStride);
        }
        return;
    }
    for (uint64_t j = j0; j < j1; ++j, v += A) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            uint32_t c = (uint32_t)__popcll(rw.w[r] ^ v);
            c = j > rw.i[r] ? c : dummy;
            lds_inc(lane_col + c * kStride);
        }
    }
}

// All codewords < 2^32.
template <int R>
__device__ void pairs_w1(uint32_t *lane_col, const Rows<R> &rw, uint64_t A, uint64_t j0, uint64_t j1) {
    uint32_t w[R];
#pragma unroll
    for (int r = 0; r < R; ++r) w[r] = (uint32_t)rw.w[r];
    const uint32_t a = (uint32_t)A;
    uint32_t v = uniform32((uint32_t)(A * j0));
    uint32_t n = uniform32((uint32_t)(j1 - j0));  // items span < 2^32 columns
    for (; n >= kUnroll; n -= kUnroll) {
#pragma unroll
        for (uint32_t u = 0; u < kUnroll; ++u) {
#pragma unroll
            for (int r = 0; r < R; ++r) lds_inc(lane_col + __popc(w[r] ^ v) * kStride);
            v += a;
        }
    }
    for (; n; --n) {
#pragma unroll
        for (int r = 0; r < R; ++r) lds_inc(lane_col + __popc(w[r] ^ v) * kStride);
        v += a;
    }
}

// 64-bit codewords, A < 2^32: within a segment of columns the high dword of
// A*j is constant, so its distance to each row's high dword is computed once
// per segment and fed to v_bcnt as the accumulate operand.
template <int R>
__device__ void pairs_w2seg(uint32_t *lane_col, const Rows<R> &rw, uint64_t A, uint64_t j0, uint64_t j1) {
    uint32_t wlo[R], whi[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        wlo[r] = (uint32_t)rw.w[r];
        whi[r] = (uint32_t)(rw.w[r] >> 32);
    }
    const uint32_t a = (uint32_t)A;
    uint64_t j = j0;
    while (j < j1) {
        const uint64_t v64 = uniform64(A * j);
        const uint32_t vhi = (uint32_t)(v64 >> 32);
        uint64_t je = j1;
        if (vhi != 0xFFFFFFFFu) {
            // first column whose high dword exceeds vhi
            const uint64_t next = ((((uint64_t)vhi + 1) << 32) + A - 1) / A;
            if (next < je) je = next;
        }
        je = uniform64(je);
        uint32_t cr[R];
#pragma unroll
        for (int r = 0; r < R; ++r) cr[r] = __popc(whi[r] ^ vhi);
        uint32_t v = (uint32_t)v64;
        uint32_t n = uniform32((uint32_t)(je - j));
        for (; n >= kUnroll; n -= kUnroll) {
#pragma unroll
            for (uint32_t u = 0; u < kUnroll; ++u) {
#pragma unroll
                for (int r = 0; r < R; ++r) lds_inc(lane_col + (__popc(wlo[r] ^ v) + cr[r]) * kStride);
                v += a;
            }
        }
        for (; n; --n) {
#pragma unroll
            for (int r = 0; r < R; ++r) lds_inc(lane_col + (__popc(wlo[r] ^ v) + cr[r]) * kStride);
            v += a;
        }
        j = je;
    }
}

// 64-bit codewords whose high dwords change from column to column: per pair,
// two XORs, two bit counts and the address, 5 VALU instructions, bounded
// pairs_w2gen at 6.4e12 pairs/s.  Here the matrix cores deliver the LDS addresses:
// with a row's bits as +-2 and a column's as -+64,
//   lane_address + 128 * 64 + sum over 64 bits = lane_address + 256 * distance,
// the byte address of the pair's counter, so a pair costs its LDS increment alone,
// and a tile of 32 x 32 pairs two MFMAs.  (Which lane holds which pair of a
// tile does not matter, nor the order of the bits, alike for both operands.)
// Measured, A = 58659 * 4097, 1048321 words: 84.4 -> 59.5 ms, 9.25e12 pairs/s
// of the LDS's 9.5e12; 2^16 words of A = 2^23 + 1 0.40 -> 0.31 ms.
typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

// 16 bits of a word's low and high dword (the upper ones for lanes 32 .. 63) as
// bytes: `zero` for a 0, zero ^ flip for a 1.
__device__ __forceinline__ void bit_bytes(uint64_t w, uint32_t zero, uint32_t flip, v4i (&out)[2]) {
    const uint32_t shift = (threadIdx.x >> 5) * 16;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        const uint32_t x = (uint32_t)(w >> (32 * s)) >> shift;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint32_t t = (((x >> (4 * q)) & 15u) * 0x204081u) & 0x01010101u;
            out[s][q] = (int)((((t << 8) - t) & flip) ^ zero);
        }
    }
}

// Columns [j0, j0 + 32 n) against 64 R full rows from row0.
template <int R>
__device__ void pairs_wide(uint32_t *lds, uint64_t A, uint64_t row0, uint64_t j0, uint32_t n) {
    constexpr int T = R < 4 ? 2 * R : 8;  // row tiles held at a time
    const uint32_t l = threadIdx.x & 31;
    v16i c;
#pragma unroll
    for (int e = 0; e < 16; ++e) c[e] = (int)(threadIdx.x * 4 + 128 * 64);
    for (uint32_t p = 0; p < 2 * R; p += T) {
        v4i rows[T][2];
#pragma unroll
        for (int t = 0; t < T; ++t) bit_bytes(A * (row0 + 32 * (p + t) + l), 0x02020202u, 0xFCFCFCFCu, rows[t]);
        uint64_t v = A * (j0 + l);
        for (uint32_t q = 0; q < n; ++q, v += 32 * A) {
            v4i col[2];
            bit_bytes(v, 0xC0C0C0C0u, 0x80808080u, col);
#pragma unroll
            for (int t = 0; t < T; ++t) {
                v16i d = __builtin_amdgcn_mfma_i32_32x32x32_i8(rows[t][0], col[0], c, 0, 0, 0);
                d = __builtin_amdgcn_mfma_i32_32x32x32_i8(rows[t][1], col[1], d, 0, 0, 0);
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    lds_inc(reinterpret_cast<uint32_t *>(reinterpret_cast<char *>(lds) + (uint32_t)d[e]));
            }
        }
    }
}

// The same pair by pair: the columns that fill no tile.
template <int R>
__device__ void pairs_w2gen(uint32_t *lane_col, const Rows<R> &rw, uint64_t A, uint64_t j0, uint64_t j1) {
    uint64_t v = uniform64(A * j0);
    for (uint32_t n = uniform32((uint32_t)(j1 - j0)); n; --n) {
#pragma unroll
        for (int r = 0; r < R; ++r) lds_inc(lane_col + __popcll(rw.w[r] ^ v) * kStride);
        v += A;
    }
}

__global__ void fill_zero_kernel(unsigned long long *p, size_t n) {
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        p[i] = 0;
}

// WIDE: also the code for kModeWide, whose tiles take 130 to 170 registers (3
// waves a SIMD, which is what keeps the LDS busiest: 9.25e12 pairs/s, 9.0 to
// 9.1 with 4); with it in one kernel the narrow codes lost 2 to 6 %.
// 16 rows a lane: scheduled for the 4 waves a SIMD that its registers leave (the
// compiler otherwise aims at 5 and misses them).  Measured with 16 rows: 1000
// words 0.36 -> 0.32 ms, 65537 words of A = 58659 0.61 -> 0.55, 80001 0.67 -> 0.62,
// 16384 codes of 256 words 0.92 -> 0.89.
template <int R, bool WIDE>
__global__ __launch_bounds__(64)
__attribute__((amdgpu_waves_per_eu(WIDE ? 3 : R == 16 ? 4 : 1, !WIDE && R == 16 ? 4 : 8)))
void pair_kernel(const PairJob *__restrict__ jobs, uint32_t njobs, uint64_t total_items,
                 unsigned long long *__restrict__ counter, uint32_t heads, uint32_t lds_rows) {
    extern __shared__ uint32_t lds[];
    const uint32_t lane = threadIdx.x;
    lds_clear(lds, lds_rows);
    uint32_t *const lane_col = lds + lane;
    const uint32_t dummy = lds_rows - 1;
    constexpr uint64_t RB = 64ull * R;

    uint32_t cur = 0xFFFFFFFFu;  // job whose counts sit in LDS
    uint64_t pending = 0;        // columns accumulated since the last flush

    for (uint64_t t = first_item(); t < total_items;
         t = counter ? following_item_of(counter, heads) : t + gridDim.x) {
        // job lookup: current job first, else binary search over item_begin
        uint32_t jb;
        if (cur != 0xFFFFFFFFu && t >= jobs[cur].item_begin && t < jobs[cur].item_begin + jobs[cur].items) {
            jb = cur;
        } else {
            uint32_t lo = 0, hi = njobs - 1;
            while (lo < hi) {
                const uint32_t mid = (lo + hi + 1) >> 1;
                if (jobs[mid].item_begin <= t) lo = mid; else hi = mid - 1;
            }
            jb = uniform32(lo);
        }
        const PairJob &job = jobs[jb];
        const uint64_t A = job.A, N = job.N, NC = job.NC, Q = job.Q;
        const uint64_t tl = t - job.item_begin + job.item_offset;
        // row block: largest b with prefix(b) <= tl
        uint64_t lo = 0, hi = job.T - 1;
        while (lo < hi) {
            const uint64_t mid = (lo + hi + 1) >> 1;
            if (pair_prefix(mid, NC, Q) <= tl) lo = mid; else hi = mid - 1;
        }
        const uint64_t b = uniform64(lo);
        const uint64_t c = (Q == 1 ? b : b / Q) + (tl - pair_prefix(b, NC, Q));
        const uint64_t CW = Q * RB;
        const uint64_t row0 = b * RB, row_end = row0 + RB;
        uint64_t j0 = c * CW;
        if (j0 < row0) j0 = row0;
        uint64_t j1 = (c + 1) * CW;
        if (j1 > N) j1 = N;
        j0 = uniform64(j0);
        j1 = uniform64(j1);

        if (jb != cur || (pending + (j1 - j0)) * R >= 0xFFFFFFFFull) {
            if (cur != 0xFFFFFFFFu)
                flush_rows(lds, 0, jobs[cur].nbins, hist_copy(jobs[cur].out, jobs[cur].nbins, jobs[cur].out_copies));
            cur = jb;
            pending = 0;
        }
        pending += j1 - j0;

        Rows<R> rw;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            rw.i[r] = row0 + (uint64_t)r * 64 + lane;
            rw.w[r] = A * rw.i[r];
        }
        const uint64_t jd1 = j1 < row_end ? j1 : row_end;
        if (j0 < jd1) pairs_masked<R>(lane_col, rw, A, j0, jd1, dummy);
        const uint64_t jr0 = j0 > row_end ? j0 : row_end;
        if (jr0 < j1) {
            if (job.mode == kModeW1)
                pairs_w1<R>(lane_col, rw, A, jr0, j1);
            else if (job.mode == kModeW2Seg)
                pairs_w2seg<R>(lane_col, rw, A, jr0, j1);
            else {
                const uint32_t tiles = WIDE ? uniform32((uint32_t)(j1 - jr0) / 32) : 0;
                if (WIDE) pairs_wide<R>(lds, A, row0, jr0, tiles);
                pairs_w2gen<R>(lane_col, rw, A, jr0 + 32ull * tiles, j1);
            }
        }
    }
    if (cur != 0xFFFFFFFFu)
        flush_rows(lds, 0, jobs[cur].nbins, hist_copy(jobs[cur].out, jobs[cur].nbins, jobs[cur].out_copies));
}

template <int R>
const void *pair_kernel_ptr(bool wide) {
    return wide ? reinterpret_cast<const void *>(&pair_kernel<R, true>)
                : reinterpret_cast<const void *>(&pair_kernel<R, false>);
}

const void *pair_kernel_for(uint32_t R, bool wide) {
    switch (R) {
    case 2: return pair_kernel_ptr<2>(wide);
    case 4: return pair_kernel_ptr<4>(wide);
    case 8: return pair_kernel_ptr<8>(wide);
    case 16: return pair_kernel_ptr<16>(wide);
    default: return nullptr;
    }
}

}  // namespace

uint32_t pair_max_distance(uint64_t A, uint64_t N) {
    const unsigned __int128 m = (unsigned __int128)(N - 1) * A;
    uint32_t bits = 0;
    for (unsigned __int128 x = m; x; x >>= 1) ++bits;
    return bits;
}

uint32_t pair_mode(uint64_t A, uint64_t N) {
    const uint32_t bits = pair_max_distance(A, N);
    if (bits <= 32) return kModeW1;
    // high dword of A*j stays constant for about 2^32/A consecutive columns
    // (at A = 2^22 both modes run at 9.25e12 pairs/s)
    if (A <= (1ull << 22)) return kModeW2Seg;
    return kModeWide;
}

void pair_job_geometry(PairJob &job, uint32_t R, uint32_t Q) {
    const uint64_t RB = 64ull * R;
    job.T = (job.N + RB - 1) / RB;
    if (Q == 0) Q = 1;
    job.Q = Q;
    const uint64_t CW = (uint64_t)Q * RB;
    job.NC = (job.N + CW - 1) / CW;
    job.items = pair_prefix(job.T, job.NC, job.Q);
}

uint32_t pair_waves_per_cu(uint32_t R, uint32_t lds_rows, bool wide) {
    // one occupancy query per (R, rows, kernel): the answer is a property of the
    // kernel and of gfx950's CU, the only target
    static std::atomic<uint32_t> caches[2][17][67];
    const void *k = pair_kernel_for(R, wide);
    if (!k || lds_rows > 66) return 0;
    auto &cache = caches[wide];
    const uint32_t hit = cache[R][lds_rows].load(std::memory_order_relaxed);
    if (hit) return hit;
    int blocks = 0;
    const size_t lds = (size_t)lds_rows * kStride * sizeof(uint32_t);
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, k, 64, lds) != hipSuccess) return 0;
    cache[R][lds_rows].store((uint32_t)blocks, std::memory_order_relaxed);
    return (uint32_t)blocks;
}

cr_status fill_zero_u64(unsigned long long *p, size_t n, hipStream_t stream) {
    if (n == 0) return CR_OK;
    const uint32_t threads = 256;
    uint32_t blocks = (uint32_t)((n + threads - 1) / threads);
    if (blocks > 1024) blocks = 1024;
    hipLaunchKernelGGL(fill_zero_kernel, dim3(blocks), dim3(threads), 0, stream, p, n);
    CR_HIP(hipGetLastError());
    return CR_OK;
}

cr_status launch_pairs(const PairJob *d_jobs, uint32_t njobs, uint64_t total_items, unsigned long long *counter,
                       const PairLaunchConfig &cfg, int cus, hipStream_t stream, hipEvent_t ev0, hipEvent_t ev1) {
    const void *k = pair_kernel_for(cfg.R, cfg.wide);
    if (!k) return fail(CR_ERR_INVALID_ARGUMENT, "rows_per_lane must be 2, 4, 8 or 16 (got %u)", cfg.R);
    if (cfg.lds_rows < 2 || cfg.lds_rows > 66)
        return fail(CR_ERR_INVALID_ARGUMENT, "histogram rows %u outside [2, 66]", cfg.lds_rows);
    if (njobs == 0) return fail(CR_ERR_INVALID_ARGUMENT, "no jobs");
    uint32_t waves = cfg.waves;
    if (waves == 0) {
        const uint32_t per_cu = pair_waves_per_cu(cfg.R, cfg.lds_rows, cfg.wide);
        if (per_cu == 0) return fail(CR_ERR_DEVICE, "occupancy query failed for the pair kernel");
        waves = per_cu * (uint32_t)cus;
    }
    if ((uint64_t)waves > total_items) waves = (uint32_t)(total_items ? total_items : 1);
    const size_t lds = (size_t)cfg.lds_rows * kStride * sizeof(uint32_t);
    if (cfg.allow_static && total_items > 0) {
        // at most one wave per CU less than the resident capacity, each
        // taking the same number of items
        counter = nullptr;
        const uint32_t per_cu = pair_waves_per_cu(cfg.R, cfg.lds_rows, cfg.wide);
        const uint64_t cap = (uint64_t)(per_cu > 1 ? per_cu - 1 : 1) * cus;
        if (waves > cap) waves = (uint32_t)cap;
        const uint64_t per = (total_items + waves - 1) / waves;
        waves = (uint32_t)((total_items + per - 1) / per);
    }
    // a head without a wave would keep its items: the caller may ask for fewer waves
    const uint32_t heads = std::min(cfg.heads, waves);
    if (cfg.zero_counter && counter) CR_TRY(fill_zero_u64(counter, heads > 1 ? kQueues * kQueuePitch : 1, stream));
    if (ev0) CR_HIP(hipEventRecord(ev0, stream));
    const PairJob *a_jobs = d_jobs;
    uint32_t a_njobs = njobs, a_heads = heads, a_rows = cfg.lds_rows;
    uint64_t a_items = total_items;
    unsigned long long *a_counter = counter;
    void *args[] = {(void *)&a_jobs, (void *)&a_njobs, (void *)&a_items, (void *)&a_counter, (void *)&a_heads,
                    (void *)&a_rows};
    CR_HIP(hipLaunchKernel(k, dim3(waves), dim3(64), args, lds, stream));
    if (ev1) CR_HIP(hipEventRecord(ev1, stream));
    return CR_OK;
}

}  // namespace cr
