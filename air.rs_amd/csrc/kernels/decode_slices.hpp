// The balanced-slice work division shared by the decode kernels (described at
// paged_decode_mfma.hip): the batch's 16-token tiles numbered sequence after
// sequence, cut into equal contiguous slices, one wave each.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "decode_common.hpp"
#include "decode_plan.hpp"

namespace airkv {

constexpr int kSliceThreads = 256;         // threads of every workgroup that calls these

// Reductions across the lanes 16 and 32 apart with the gfx950 lane-swap
// instructions instead of LDS permutes.  permlane16_swap(v, v) returns
// {v[l & ~16], v[l | 16]} in lane l, permlane32_swap(v, v) returns
// {v[l & ~32], v[l | 32]}: the two halves of each pair, in the same order
// in both lanes, so both lanes compute the same bits.
__device__ __forceinline__ float max_x16(float x) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float max_x32(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float sum_x16(float x) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float sum_x32(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Register-pair transposes: afterwards x_b in lane l holds what x_c held in
// lane l', where c is lane l's bit 3 (bit 5) and l' is l with that bit set
// to b.  Bit 3: DPP row_ror:8 (lane l ^ 8 within each row of 16), written
// only to the lanes whose bit 3 differs from the register index (bank masks
// 0xC: lanes 8..15 of each row, 0x3: lanes 0..7).  Bit 5: the lane swap
// across the wave's halves.
__device__ __forceinline__ void swap_lane_bit3(u32x4 &x0, u32x4 &x1) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int a = (int)x0[j], b = (int)x1[j];
        x0[j] = (uint32_t)__builtin_amdgcn_update_dpp(a, b, 0x128, 0xF, 0xC, false);
        x1[j] = (uint32_t)__builtin_amdgcn_update_dpp(b, a, 0x128, 0xF, 0x3, false);
    }
}
__device__ __forceinline__ void swap_lane_bit5(u32x4 &x0, u32x4 &x1) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const auto r = __builtin_amdgcn_permlane32_swap(x0[j], x1[j], false, false);
        x0[j] = r[0];
        x1[j] = r[1];
    }
}

__device__ __forceinline__ int64_t clamp_len(int64_t len, int64_t max_len) {
    return len < 0 ? 0 : (len > max_len ? max_len : len);
}

// Inclusive sum / running maximum over a wave's lanes (DPP: row shifts, then
// the rows' last lanes broadcast; the identity of both is 0).
template <class F> __device__ __forceinline__ int wave_scan(int x, F f) {
    x = f(x, __builtin_amdgcn_update_dpp(0, x, 0x111, 0xF, 0xF, false));   // row_shr:1
    x = f(x, __builtin_amdgcn_update_dpp(0, x, 0x112, 0xF, 0xF, false));   // row_shr:2
    x = f(x, __builtin_amdgcn_update_dpp(0, x, 0x114, 0xF, 0xF, false));   // row_shr:4
    x = f(x, __builtin_amdgcn_update_dpp(0, x, 0x118, 0xF, 0xF, false));   // row_shr:8
    x = f(x, __builtin_amdgcn_update_dpp(0, x, 0x142, 0xA, 0xF, false));   // row_bcast:15 into rows 1, 3
    x = f(x, __builtin_amdgcn_update_dpp(0, x, 0x143, 0xC, 0xF, false));   // row_bcast:31 into rows 2, 3
    return x;
}

// pre[b] = tiles (ceil(len / 16), len clamped to [0, max_blocks * bs]) of the
// sequences before b, for b = 0..batch, in LDS, and pre[B + 1] = the most
// tiles of one sequence.  All threads take part.
// long_seq (optional, ceil(B / 32) words): bit b set when sequence b is longer
// than its table, else clear.
//
// Up to kScanBatch sequences: every wave scans them in registers, 64 at a time,
// and writes the same values, which it alone reads, so the launch's first loads
// are not held up by the workgroup's barriers.
__device__ __forceinline__ void tile_prefix(const DecodeArgs &a, int bs, int32_t *pre, int32_t *wsum,
                                            uint32_t *long_seq = nullptr) {
    constexpr int kScanBatch = 256, kSteps = kScanBatch / 64;
    if (a.batch <= kScanBatch) {
        const int lane = threadIdx.x & 63, B = a.batch;
        const int64_t max_len = (int64_t)a.max_blocks * bs;
        int32_t len[kSteps];
#pragma unroll
        for (int k = 0; k < kSteps; ++k) len[k] = 64 * k + lane < B ? a.lens[64 * k + lane] : 0;
        int before = 0, most = 0;
#pragma unroll
        for (int k = 0; k < kSteps; ++k) {
            if (64 * k >= B) break;
            const int32_t t = (int32_t)((clamp_len(len[k], max_len) + 15) / 16);
            const int incl = before + wave_scan(t, [](int x, int y) { return x + y; });
            if (64 * k + lane < B) pre[64 * k + lane + 1] = incl;
            before = __builtin_amdgcn_readlane(incl, 63);
            most = max(most, t);
            if (long_seq) {
                const uint64_t m = __ballot(len[k] > max_len);
                if (lane < 2 && 64 * k + 32 * lane < B) long_seq[2 * k + lane] = (uint32_t)(lane ? m >> 32 : m);
            }
        }
        most = wave_scan(most, [](int x, int y) { return x > y ? x : y; });
        if (lane == 63) {
            pre[0] = 0;
            pre[B + 1] = most;
        }
        // lanes read what other lanes of their wave wrote: LDS serves a wave in
        // order, this keeps the compiler from moving a read ahead of the writes
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        return;
    }
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int B = a.batch;
    const int64_t max_len = (int64_t)a.max_blocks * bs;
    if (long_seq) {
        for (int i = tid; i < (B + 31) / 32; i += kSliceThreads) long_seq[i] = 0;
        __syncthreads();
    }
    int tmax = 0;
    for (int b = tid; b < B; b += kSliceThreads) {
        const int32_t len = a.lens[b];
        const int32_t t = (int32_t)((clamp_len(len, max_len) + 15) / 16);
        pre[b + 1] = t;
        tmax = t > tmax ? t : tmax;
        if (long_seq && len > max_len) atomicOr(&long_seq[b >> 5], 1u << (b & 31));
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const int y = __shfl_xor(tmax, o);
        tmax = y > tmax ? y : tmax;
    }
    if (lane == 0) wsum[wave] = tmax;
    if (tid == 0) pre[0] = 0;
    __syncthreads();
    if (tid == 0) {
        int m = wsum[0];
        for (int w = 1; w < kSliceThreads / 64; ++w) m = wsum[w] > m ? wsum[w] : m;
        pre[B + 1] = m;
    }
    __syncthreads();
    // each thread scans a run of `per` entries; runs are chained by a
    // wave-level then a workgroup-level exclusive scan of the run sums
    const int per = (B + kSliceThreads - 1) / kSliceThreads;
    const int lo = 1 + tid * per;
    const int hi = lo + per < B + 1 ? lo + per : B + 1;
    int sum = 0;
    for (int i = lo; i < hi; ++i) sum += pre[i];
    int incl = sum;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(incl, o);
        if (lane >= o) incl += y;
    }
    if (lane == 63) wsum[wave] = incl;
    __syncthreads();
    int run = incl - sum;
    for (int w = 0; w < wave; ++w) run += wsum[w];
    for (int i = lo; i < hi; ++i) {
        run += pre[i];
        pre[i] = run;
    }
    __syncthreads();
}

// The sequence holding tile t (0 <= t < pre[B]): the b with pre[b] <= t < pre[b + 1].
// The loop count depends on B only, so the lanes of a wave stay converged.
__device__ __forceinline__ int seq_of_tile(const int32_t *pre, int B, int t) {
    int lo = 0, hi = B;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (pre[mid] <= t) lo = mid;
        else hi = mid;
    }
    return lo;
}

}  // namespace airkv
