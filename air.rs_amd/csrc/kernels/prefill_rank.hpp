// Device helpers shared by the prefill kernels: the consistency test of a
// sequence, the setup of a workgroup and the ranking of a launch's work items
// by length.
#pragma once

#include <hip/hip_runtime.h>

#include "air_kv.h"
#include "prefill_common.hpp"

namespace airkv {

constexpr int kRankThreads = 256;           // threads of every workgroup that calls these
constexpr int kRankWaves = kRankThreads / 64;
constexpr int kRankCap = 2048;
constexpr int kRankItems = 64 * kRankThreads;
constexpr int kRankLdsBytes = (kRankThreads + kRankWaves + 8 + 2 * kRankCap) * 4;

// Whether sequence b's rows and length are consistent: 0 <= cu_q[b] <=
// cu_q[b + 1] <= total_q, 0 <= seq_len <= max_blocks * block_size and
// q_len <= seq_len.  The one test every prefill kernel applies: an
// inconsistent sequence is counted and zero-filled by its first workgroup,
// never split into pieces and never written by the merge.
__device__ __forceinline__ bool prefill_rows_ok(const PrefillArgs &a, int b) {
    const int32_t q0 = a.cu_q[b], q1 = a.cu_q[b + 1];
    return q0 >= 0 && q1 >= q0 && q1 <= a.total_q;
}
__device__ __forceinline__ bool prefill_seq_ok(const PrefillArgs &a, int b) {
    const int64_t len = a.lens[b];
    const int64_t qlen = (int64_t)a.cu_q[b + 1] - a.cu_q[b];
    return prefill_rows_ok(a, b) && len >= 0 && len <= a.max_len && qlen <= len;
}

// Per-(sequence, kv head) setup shared by the prefill kernels: reads the
// sequence's rows and length, counts (once) an inconsistent sequence,
// zero-fills its rows, and returns whether the workgroup has rows to compute.
// Uniform per workgroup.  `first`: the sequence's first workgroup of this kv
// head; d: the pool's head_dim.
__device__ __forceinline__ bool prefill_begin(const PrefillArgs &a, int b, int kh, bool first, int d, int32_t &q0,
                                              int &qlen, int64_t &len) {
    const int tid = threadIdx.x;
    const int G = a.group;
    q0 = a.cu_q[b];
    len = a.lens[b];
    qlen = a.cu_q[b + 1] - q0;
    if (prefill_seq_ok(a, b)) return qlen > 0;
    if (first && kh == 0 && tid == 0) atomicAdd(a.errors, 1ull);
    // rows of a sequence whose lengths are inconsistent become zeros
    if (first && prefill_rows_ok(a, b)) {
        const int64_t n = (int64_t)qlen * G * d;
        for (int64_t i = tid; i < n; i += kRankThreads) {
            const int64_t r = i / (G * d), e = i % (G * d);
            const int64_t idx = ((int64_t)(q0 + r) * a.n_q_heads + kh * G) * d + e;
            if (a.out_dtype == AIR_KV_F32) ((float *)a.out)[idx] = 0.0f;
            else ((uint16_t *)a.out)[idx] = 0;
        }
    }
    return false;
}

// Counts the out-of-pool table entries within sequence b's length (once per
// sequence that has query rows: one workgroup calls this).
__device__ __forceinline__ void prefill_count_entries(const PrefillArgs &a, int b, int bs, int64_t len) {
    const int32_t *tbl = a.tables + (int64_t)b * a.max_blocks;
    for (int64_t j = threadIdx.x; j < (len + bs - 1) / bs; j += kRankThreads) {
        const int32_t blk = tbl[j];
        if (blk < 0 || blk >= a.num_blocks) atomicAdd(a.errors, 1ull);
    }
}

__device__ __forceinline__ int len_bucket(int64_t len) {   // 0 .. 248, monotone in len
    if (len <= 0) return 0;
    const uint32_t x = len > 0x7fffffff ? 0x7fffffffu : (uint32_t)len;
    const int e = 31 - __builtin_clz(x);
    const int m = e >= 3 ? (int)(x >> (e - 3)) & 7 : (int)(x << (3 - e)) & 7;
    return 1 + 8 * e + m;
}

// Exclusive prefix sum over the workgroup's threads in thread order; wsum
// holds kRankWaves ints of LDS.  Contains barriers: every thread calls it.
__device__ __forceinline__ int block_exclusive_scan(int v, int *wsum) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int incl = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(incl, o);
        if (lane >= o) incl += y;
    }
    if (lane == 63) wsum[wave] = incl;
    __syncthreads();
    int base = 0;
    for (int w = 0; w < wave; ++w) base += wsum[w];
    __syncthreads();
    return base + incl - v;
}

// The (sequence, slot) item of rank `row`, item = sequence * nz + slot, when
// the batch * nz items (at most kRankItems, batch at most kRankCap) are
// ordered by keys(seq_len, q_len, slot), decreasing, in buckets of an eighth
// of an octave, ties by index.  lds: kRankLdsBytes, free for the duration and
// on return.  Every thread calls it.
template <class Keys>
__device__ __forceinline__ int rank_item(const PrefillArgs &a, int *lds, int nz, int row, Keys keys) {
    const int tid = threadIdx.x;
    int *hist = lds, *wsum = lds + kRankThreads, *sel = lds + kRankThreads + kRankWaves;
    int *slen = sel + 8, *sq = slen + kRankCap;
    hist[tid] = 0;
    for (int i = tid; i < a.batch; i += kRankThreads) {
        slen[i] = a.lens[i];
        const int64_t ql = (int64_t)a.cu_q[i + 1] - a.cu_q[i];
        sq[i] = ql < 0 ? 0 : ql > 0x7fffffff ? 0x7fffffff : (int)ql;
    }
    __syncthreads();
    const int n_it = a.batch * nz;
    const int chunk = (n_it + kRankThreads - 1) / kRankThreads;
    const int i0 = tid * chunk, i1 = i0 + chunk < n_it ? i0 + chunk : n_it;
    auto bucket_of = [&](int i) {
        const int bb = i / nz;
        return len_bucket(keys(slen[bb], sq[bb], i - bb * nz));
    };
    for (int i = i0; i < i1; ++i) atomicAdd(&hist[bucket_of(i)], 1);
    __syncthreads();
    // buckets in decreasing order: thread t takes bucket kRankThreads - 1 - t
    const int bucket = kRankThreads - 1 - tid;
    const int cnt = hist[bucket];
    const int start = block_exclusive_scan(cnt, wsum);
    if (row >= start && row < start + cnt) {
        sel[0] = bucket;
        sel[1] = row - start;
    }
    __syncthreads();
    const int want = sel[0], j = sel[1];
    // the j-th item (index order) of bucket want: thread t scans its chunk
    int c = 0;
    for (int i = i0; i < i1; ++i) c += bucket_of(i) == want;
    const int before = block_exclusive_scan(c, wsum);
    if (j >= before && j < before + c) {
        int k = j - before;
        for (int i = i0; i < i1; ++i)
            if (bucket_of(i) == want && k-- == 0) sel[0] = i;
    }
    __syncthreads();
    const int item = sel[0];
    __syncthreads();   // the caller reuses the LDS
    return item;
}

}  // namespace airkv
