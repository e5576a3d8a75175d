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

// A workgroup's place in a launch.
struct PrefillSlot {
    int b, kh, z, nz;          // sequence, kv head, slot of it, slots per sequence
    int p, ns, ord;            // piece, pieces of the slot (1: not split), split ordinal (-1: none)
};

// Per-(sequence, kv head) setup shared by the prefill kernels: reads the
// sequence's rows and length, counts (once) an inconsistent sequence and, with
// BS > 0 (the block size), every out-of-pool table entry within its length
// (else the caller counts them), zero-fills the rows of an inconsistent
// sequence, and returns whether the workgroup has rows to compute.  Uniform
// per workgroup.  D: the head_dim (0: the pool's, read from the arguments).
// The table loop is written out here: as a function of its own it changed the
// matrix-core kernel's register allocation (six int8 chunks of up to 512 tokens
// over up to 6000, 64 heads over 8: 437.8 us, 435.3 this way).
template <int BS, int D>
__device__ bool prefill_begin(const PrefillArgs &a, const PrefillSlot &sl, int32_t &q0, int &qlen, int64_t &len) {
    const int b = sl.b, kh = sl.kh, tid = threadIdx.x;
    const int G = a.group, d = D ? D : a.head_dim;
    q0 = a.cu_q[b];
    len = a.lens[b];
    qlen = a.cu_q[b + 1] - q0;
    const bool rows_ok = prefill_rows_ok(a, b);
    const bool seq_ok = prefill_seq_ok(a, b);
    const int32_t *tbl = a.tables + (int64_t)b * a.max_blocks;
    if (sl.z == 0 && sl.p == 0 && kh == 0) {
        if (!seq_ok) {
            if (tid == 0) atomicAdd(a.errors, 1ull);
        } else if (qlen > 0) {
            if constexpr (BS > 0) {
                for (int64_t j = tid; j < (len + BS - 1) / BS; j += kRankThreads) {
                    const int32_t blk = tbl[j];
                    if (blk < 0 || blk >= a.num_blocks) atomicAdd(a.errors, 1ull);
                }
            }
        }
    }
    if (!seq_ok) {
        // rows of a sequence whose lengths are inconsistent become zeros
        if (rows_ok && sl.z == 0 && sl.p == 0) {
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
    return qlen > 0;
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
