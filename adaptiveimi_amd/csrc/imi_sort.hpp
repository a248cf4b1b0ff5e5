// Device building blocks of the stable counting sorts: a superblock's items
// put in digit order by one workgroup, and an exclusive scan.  Used for the
// k-means member lists (digit = subspace label) and for the LSD cell sort (one
// pass per subspace label), which reproduces the reference's ascending-token
// counting sort (reorganize_core.cpp:287-295).
#pragma once

#include <algorithm>

#include "imi_common.hpp"

namespace imi {

// Intra-wave LDS hand-off (compiler ordering only; a wave's LDS instructions
// execute in order).
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__host__ __device__ inline int bits_for(int n) {
    int b = 0;
    while ((1 << b) < n) ++b;
    return b;
}

// Superblocks of T items in `segs` independent rows: about two rounds of
// workgroups over the device, 1024 .. 8192 items each (a superblock then sorts
// in LDS), and at most kMaxSuper of them.
constexpr int kMaxSuper = 512;
constexpr int kStagedItems = 32768;   // items per superblock up to which the order is staged in LDS

inline void superblocks(int T, int segs, int& items, int& count) {
    items = 1024;
    while (items < 8192 && static_cast<int64_t>(items) * 2 * device_cus() < static_cast<int64_t>(T) * segs) items *= 2;
    while ((static_cast<int64_t>(T) + items - 1) / items > kMaxSuper) items *= 2;
    count = static_cast<int>((static_cast<int64_t>(T) + items - 1) / items);
}

// Waves per workgroup: 16, but 4 where the label counts per wave would not
// leave room in LDS.
inline int sort_waves(int kmax) { return kmax <= 512 ? 16 : 4; }

// Stable counting sort of a superblock of m <= items items (items / waves a
// multiple of 64) by digit(i) in [0, k): item counts per wave (a wave owns
// consecutive items), one scan over (digit, wave), then every round of 64
// items takes its places from the wave's running offsets.  row(c, first)
// receives each digit's first place, place(i, at) each item's.  cnt: LDS of
// waves x k ints, wsum of 16.  All threads of the workgroup; ends without a
// barrier after the last place().
template <typename Digit, typename Row, typename Place>
__device__ __forceinline__ void superblock_sort(int m, int items, int k, int* cnt, int* wsum, Digit digit, Row row,
                                                Place place) {
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int nthr = blockDim.x, nw = nthr >> 6;
    const int span = items / nw;
    const int w0 = wave * span, w1 = min(w0 + span, m);
    const int bits = bits_for(k);
    for (int i = tid; i < nw * k; i += nthr) cnt[i] = 0;
    __syncthreads();
    int* mine = cnt + wave * k;
    for (int i = w0; i < w1; i += 256) {
        int l[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) l[u] = digit(min(i + 64 * u + lane, m - 1));
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (i + 64 * u + lane < w1) atomicAdd(&mine[l[u]], 1);
    }
    __syncthreads();
    // exclusive offsets over (digit, wave): consecutive digits per thread
    const int per = (k + nthr - 1) / nthr;
    const int c0 = min(tid * per, k), c1 = min(c0 + per, k);
    int local = 0;
    for (int c = c0; c < c1; ++c)
        for (int w = 0; w < nw; ++w) local += cnt[w * k + c];
    const int incl = wave_incl_scan(local);
    if (lane == 63) wsum[wave] = incl;
    __syncthreads();
    int run = incl - local;
    for (int w = 0; w < wave; ++w) run += wsum[w];
    for (int c = c0; c < c1; ++c) {
        row(c, run);
        for (int w = 0; w < nw; ++w) {
            const int n = cnt[w * k + c];
            cnt[w * k + c] = run;
            run += n;
        }
    }
    __syncthreads();
    for (int i = w0; i < w1; i += 256) {
        int l[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) l[u] = digit(min(i + 64 * u + lane, m - 1));
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if (i + 64 * u >= w1) break;
            const int it = i + 64 * u + lane;
            const bool in = it < w1;
            const uint64_t peers = match_peers(static_cast<uint32_t>(l[u]), bits, __ballot(in));
            const int rank = __popcll(peers & lanemask_lt());
            const int at = in ? mine[l[u]] : 0;
            wave_lds_order();
            if (in) {
                if (rank == 0) mine[l[u]] = at + __popcll(peers);
                place(it, at + rank);
            }
            wave_lds_order();
        }
    }
}

// Exclusive scan, in place, of n ints by one 1024-thread block.  `sh` is LDS
// of at least 33 ints.  Returns the total on every thread.  Each thread owns a
// contiguous chunk; when n is a multiple of 4 and data 16-byte aligned the
// chunks are whole int4s read 8 at a time (8 loads in flight per thread).
typedef int __attribute__((ext_vector_type(4))) scan_i32x4_t;

__device__ __forceinline__ int block_exclusive_scan_1024(int32_t* data, int64_t n, int* sh) {
    const int tid = threadIdx.x;
    const bool vec = (n % 4) == 0 && (reinterpret_cast<uintptr_t>(data) & 15) == 0;
    int64_t per = (n + 1023) / 1024;
    if (vec) per = (per + 3) & ~static_cast<int64_t>(3);
    const int64_t lo = tid * per < n ? tid * per : n;
    const int64_t hi = lo + per < n ? lo + per : n;
    int local = 0;
    if (vec) {
        for (int64_t i = lo; i < hi; i += 32) {
            scan_i32x4_t v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u)
                v[u] = i + 4 * u < hi ? *reinterpret_cast<const scan_i32x4_t*>(data + i + 4 * u)
                                      : scan_i32x4_t{0, 0, 0, 0};
#pragma unroll
            for (int u = 0; u < 8; ++u) local += (v[u][0] + v[u][1]) + (v[u][2] + v[u][3]);
        }
    } else {
        for (int64_t i = lo; i < hi; ++i) local += data[i];
    }
    const int incl = wave_incl_scan(local);
    const int wave = tid >> 6;
    if (lane_id() == 63) sh[wave] = incl;
    __syncthreads();
    if (tid < 64) {
        int v = tid < 16 ? sh[tid] : 0;
        int s = wave_incl_scan(v);
        if (tid < 16) sh[16 + tid] = s - v;
        if (tid == 15) sh[32] = s;
    }
    __syncthreads();
    int run = sh[16 + wave] + incl - local;
    if (vec) {
        for (int64_t i = lo; i < hi; i += 32) {
            scan_i32x4_t v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u)
                v[u] = i + 4 * u < hi ? *reinterpret_cast<const scan_i32x4_t*>(data + i + 4 * u)
                                      : scan_i32x4_t{0, 0, 0, 0};
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                if (i + 4 * u < hi) {
                    scan_i32x4_t o;
                    o[0] = run;
                    run += v[u][0];
                    o[1] = run;
                    run += v[u][1];
                    o[2] = run;
                    run += v[u][2];
                    o[3] = run;
                    run += v[u][3];
                    *reinterpret_cast<scan_i32x4_t*>(data + i + 4 * u) = o;
                }
            }
        }
    } else {
        for (int64_t i = lo; i < hi; ++i) {
            const int v = data[i];
            data[i] = run;
            run += v;
        }
    }
    const int total = sh[32];
    __syncthreads();
    return total;
}

}  // namespace imi
