// Paged prefill, one query row at a time on the vector units: the pools
// paged_prefill.hip does not take (f32 pages, head_dim other than 128), for
// launches too small for paged_prefill_f32.hip (prefill_f32_better).
//
// A workgroup owns one (query row, kv head, sequence) and the query heads that
// share the kv head (GQA, src/chunked_attn.rs:240-243), G of them at a time:
// groups of up to 8 heads take one workgroup per kv head (G the next power of
// two, heads past the group masked), larger groups ceil(group / G) workgroups
// of G heads each.  It runs an online softmax over the row's causal keys in
// 64-token tiles and writes the normalised output.
//
// Thread mapping: head_dim/8 lanes cover one token row, 8 elements per lane,
// loaded with one 16-byte (bf16) or 8-byte (int8/fp8) access; a 64-lane wave
// covers 512/head_dim rows per pass.  Dot products reduce across the row's
// lanes with butterfly shuffles.  Quantized pages are dequantized in
// registers (code * group scale, as the oracle's dequantized cache).
#include <hip/hip_runtime.h>

#include <cmath>

#include "../pool.hpp"
#include "codecs.hpp"
#include "prefill_common.hpp"

namespace airkv {
namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;
constexpr int kTile = 64;          // tokens per online-softmax step

// Raw storage of 8 cache elements in registers.
template <int DT> struct Raw8;
template <> struct Raw8<AIR_KV_F32> { float4 a, b; };
template <> struct Raw8<AIR_KV_BF16> { uint4 w; };
template <> struct Raw8<AIR_KV_INT8> { uint2 w; float s; };
template <> struct Raw8<AIR_KV_FP8> { uint2 w; float s; };

template <int DT>
__device__ __forceinline__ void load_raw(const void *pages, const float *scales, int64_t elem,
                                         int64_t sidx, Raw8<DT> &r) {
    if constexpr (DT == AIR_KV_F32) {
        const float4 *p = reinterpret_cast<const float4 *>((const float *)pages + elem);
        r.a = p[0];
        r.b = p[1];
    } else if constexpr (DT == AIR_KV_BF16) {
        r.w = *reinterpret_cast<const uint4 *>((const uint16_t *)pages + elem);
    } else {
        r.w = *reinterpret_cast<const uint2 *>((const uint8_t *)pages + elem);
        r.s = scales[sidx];
    }
}

template <int DT>
__device__ __forceinline__ void zero_raw(Raw8<DT> &r) {
    if constexpr (DT == AIR_KV_F32) { r.a = make_float4(0, 0, 0, 0); r.b = r.a; }
    else if constexpr (DT == AIR_KV_BF16) { r.w = make_uint4(0, 0, 0, 0); }
    else { r.w = make_uint2(0, 0); r.s = 0.0f; }
}

template <int DT>
__device__ __forceinline__ void unpack(const Raw8<DT> &r, float (&x)[8]) {
    if constexpr (DT == AIR_KV_F32) {
        x[0] = r.a.x; x[1] = r.a.y; x[2] = r.a.z; x[3] = r.a.w;
        x[4] = r.b.x; x[5] = r.b.y; x[6] = r.b.z; x[7] = r.b.w;
    } else if constexpr (DT == AIR_KV_BF16) {
        const uint32_t u[4] = {r.w.x, r.w.y, r.w.z, r.w.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            x[2 * j] = __uint_as_float(u[j] << 16);
            x[2 * j + 1] = __uint_as_float(u[j] & 0xFFFF0000u);
        }
    } else {
        const uint32_t u[2] = {r.w.x, r.w.y};
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint32_t byte = (u[j >> 2] >> (8 * (j & 3))) & 0xFFu;
            float val;
            if constexpr (DT == AIR_KV_INT8) val = (float)(int32_t)(int8_t)byte;
            else val = fp8_decode(byte);
            x[j] = val * r.s;
        }
    }
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) v = fmaxf(v, __shfl_xor(v, m));
    return v;
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m);
    return v;
}

template <int DT, int G, int DP>
__global__ __launch_bounds__(kThreads) void prefill_rows_kernel(PrefillArgs a) {
    // DP: head_dim rounded up to 64, 128 or 256 (lanes past head_dim idle).
    // G: query heads per workgroup, the group's heads g0 .. g0 + gn - 1.
    constexpr int LPR = DP / 8;                 // lanes per token row
    constexpr int RPW = 64 / LPR;               // rows per wave per pass
    constexpr int RPP = RPW * kWaves;           // rows per workgroup pass
    constexpr int PASSES = kTile / RPP;
    constexpr bool QUANT = DT == AIR_KV_INT8 || DT == AIR_KV_FP8;
    static_assert(PASSES >= 1 && kTile % RPP == 0, "tile must cover whole passes");

    __shared__ float s_p[G * kTile];
    __shared__ float s_m[G], s_l[G], s_alpha[G];
    __shared__ float s_red[(kWaves - 1) * G * DP];

    const int d = a.head_dim;
    const int chunks = (a.group + G - 1) / G;
    const int kh = blockIdx.y / chunks, g0 = (blockIdx.y % chunks) * G;
    const int gn = a.group - g0 < G ? a.group - g0 : G;   // heads of the group in this workgroup
    const int64_t head0 = (int64_t)kh * a.group + g0;       // its first query head
    const int b = blockIdx.z;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t max_len = (int64_t)a.max_blocks * a.block_size;
    const int chunk = lane % LPR;
    const bool cv = chunk * 8 < d;              // the lane's 8 elements lie inside head_dim
    const int row_in_pass = wave * RPW + lane / LPR;
    const int ng = QUANT ? d / a.scale_group : 1;
    // block sizes (16, 32) and scale groups are powers of two: the per-row
    // index arithmetic below shifts and masks instead of dividing
    const int bs_log2 = __builtin_ctz((unsigned)a.block_size);
    const int64_t bs_mask = a.block_size - 1;
    const int sg_log2 = QUANT ? __builtin_ctz((unsigned)a.scale_group) : 0;
    const int32_t *table = a.tables + (int64_t)b * a.max_blocks;

    float qr[G][8];                             // this lane's 8 elements of each query row, f32
    float acc[G][8];

    // q row `qrow` (zeros for heads past the group and lanes past head_dim)
    auto load_q = [&](int64_t qrow) {
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const int64_t qoff = (qrow * a.n_q_heads + head0 + g) * d + chunk * 8;
            if (g >= gn || !cv) {
#pragma unroll
                for (int j = 0; j < 8; ++j) qr[g][j] = 0.0f;
            } else if (a.q_dtype == AIR_KV_F32) {
                const float4 *qp = reinterpret_cast<const float4 *>((const float *)a.q + qoff);
                float4 x0 = qp[0], x1 = qp[1];
                qr[g][0] = x0.x; qr[g][1] = x0.y; qr[g][2] = x0.z; qr[g][3] = x0.w;
                qr[g][4] = x1.x; qr[g][5] = x1.y; qr[g][6] = x1.z; qr[g][7] = x1.w;
            } else {
                uint4 w = *reinterpret_cast<const uint4 *>((const uint16_t *)a.q + qoff);
                const uint32_t u[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    qr[g][2 * j] = __uint_as_float(u[j] << 16);
                    qr[g][2 * j + 1] = __uint_as_float(u[j] & 0xFFFF0000u);
                }
            }
        }
    };

    // Keys [0, end) of this workgroup's sequence: online softmax into acc
    // (unnormalised) and s_m / s_l, then acc summed over the rows of the wave
    // and over the waves, the total in wave 0's lanes < LPR.  The tokens of an
    // out-of-pool table entry read as zero keys and values; `count`: it is
    // counted, at its block's first token.
    auto attend = [&](int64_t end, bool count) {
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
            for (int j = 0; j < 8; ++j) acc[g][j] = 0.0f;
        __syncthreads();                        // the previous pass's readers of s_m / s_l / s_red
        if (tid < G) { s_m[tid] = -INFINITY; s_l[tid] = 0.0f; }
        __syncthreads();
        for (int64_t t0 = 0; t0 < end; t0 += kTile) {
            Raw8<DT> vraw[PASSES];
            // ---- scores s = q . k (log2 units) for the tile's rows
#pragma unroll
            for (int ps = 0; ps < PASSES; ++ps) {
                const int r = ps * RPP + row_in_pass;
                const int64_t t = t0 + r;
                const bool ok = t < end;
                int32_t blk = ok ? table[t >> bs_log2] : 0;
                bool in_pool = true;
                if (ok && (blk < 0 || blk >= a.num_blocks)) {
                    in_pool = false;
                    if (chunk == 0 && count && (t & bs_mask) == 0) atomicAdd(a.errors, 1ull);
                }
                Raw8<DT> kraw;
                if (ok && cv && in_pool) {
                    const int64_t row = ((int64_t)blk * a.n_kv_heads + kh) * a.block_size + (t & bs_mask);
                    const int64_t sidx = row * ng + ((chunk * 8) >> sg_log2);
                    load_raw<DT>(a.k_pages, a.k_scales, row * d + chunk * 8, sidx, kraw);
                    load_raw<DT>(a.v_pages, a.v_scales, row * d + chunk * 8, sidx, vraw[ps]);
                } else {
                    zero_raw<DT>(kraw);
                    zero_raw<DT>(vraw[ps]);
                }
                float kx[8];
                unpack<DT>(kraw, kx);
                float sc[G];
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    float s = 0.0f;
#pragma unroll
                    for (int j = 0; j < 8; ++j) s += qr[g][j] * kx[j];
                    sc[g] = s;
                }
#pragma unroll
                for (int m = LPR / 2; m >= 1; m >>= 1)
#pragma unroll
                    for (int g = 0; g < G; ++g) sc[g] += __shfl_xor(sc[g], m);
                if (chunk == 0) {
#pragma unroll
                    for (int g = 0; g < G; ++g) s_p[g * kTile + r] = ok ? sc[g] * a.scale_log2 : -INFINITY;
                }
            }
            __syncthreads();
            // ---- online softmax update, one head per wave at a time
            for (int g = wave; g < G; g += kWaves) {
                const float s = s_p[g * kTile + lane];
                const float m_old = s_m[g];
                const float m_new = fmaxf(m_old, wave_max(s));
                const float p = (s == -INFINITY) ? 0.0f : exp2f(s - m_new);
                const float psum = wave_sum(p);
                s_p[g * kTile + lane] = p;
                if (lane == 0) {
                    const float alpha = (m_old == -INFINITY) ? 0.0f : exp2f(m_old - m_new);
                    s_alpha[g] = alpha;
                    s_l[g] = s_l[g] * alpha + psum;
                    s_m[g] = m_new;
                }
            }
            __syncthreads();
            // ---- acc = acc * alpha + p . V
#pragma unroll
            for (int g = 0; g < G; ++g) {
                const float al = s_alpha[g];
#pragma unroll
                for (int j = 0; j < 8; ++j) acc[g][j] *= al;
            }
#pragma unroll
            for (int ps = 0; ps < PASSES; ++ps) {
                const int r = ps * RPP + row_in_pass;
                float vx[8];
                unpack<DT>(vraw[ps], vx);
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    const float p = s_p[g * kTile + r];
#pragma unroll
                    for (int j = 0; j < 8; ++j) acc[g][j] += p * vx[j];
                }
            }
            __syncthreads();
        }
        // ---- reduce acc over the rows of the wave, then over the waves
#pragma unroll
        for (int m = LPR; m < 64; m <<= 1)
#pragma unroll
            for (int g = 0; g < G; ++g)
#pragma unroll
                for (int j = 0; j < 8; ++j) acc[g][j] += __shfl_xor(acc[g][j], m);
        if (wave > 0 && lane < LPR) {
#pragma unroll
            for (int g = 0; g < G; ++g)
#pragma unroll
                for (int j = 0; j < 8; ++j) s_red[((wave - 1) * G + g) * DP + chunk * 8 + j] = acc[g][j];
        }
        __syncthreads();
        if (wave == 0 && lane < LPR) {
#pragma unroll
            for (int g = 0; g < G; ++g)
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    float v = acc[g][j];
#pragma unroll
                    for (int w = 0; w < kWaves - 1; ++w) v += s_red[(w * G + g) * DP + chunk * 8 + j];
                    acc[g][j] = v;
                }
        }
    };

    // Prefill rows: sequence b's query rows q0 .. q1 - 1, row r at
    // position len - q_len + r seeing keys 0 ..= that position, each a
    // single partition normalised here.  The consistency test and its
    // handling are the matrix-core prefill's: counted once, rows inside
    // [0, total_q] zero-filled.
    const int32_t q0 = a.cu_q[b], q1 = a.cu_q[b + 1];
    const int64_t len = a.lens[b];
    const bool rows_ok = q0 >= 0 && q1 >= q0 && q1 <= a.total_q;
    const int qlen = q1 - q0;
    if (!(rows_ok && len >= 0 && len <= max_len && (int64_t)qlen <= len)) {
        if (blockIdx.x == 0 && blockIdx.y == 0 && tid == 0) atomicAdd(a.errors, 1ull);
        if (!rows_ok) return;
        for (int r = blockIdx.x; r < qlen; r += gridDim.x)
            for (int i = tid; i < gn * d; i += kThreads) {
                const int64_t oi = (((int64_t)q0 + r) * a.n_q_heads + head0 + i / d) * d + i % d;
                if (a.out_dtype == AIR_KV_F32) ((float *)a.out)[oi] = 0.0f;
                else ((uint16_t *)a.out)[oi] = 0;
            }
        return;
    }
    for (int r = blockIdx.x; r < qlen; r += gridDim.x) {
        const int64_t qrow = (int64_t)q0 + r;
        load_q(qrow);
        // the last row reads every key: its first head chunk counts each
        // out-of-pool entry once
        attend(len - qlen + r + 1, r == qlen - 1 && blockIdx.y == 0);
        if (wave == 0 && lane < LPR && cv) {
#pragma unroll
            for (int g = 0; g < G; ++g) {
                if (g >= gn) break;
                const float inv = 1.0f / s_l[g];
                const int64_t oi = (qrow * a.n_q_heads + head0 + g) * d + chunk * 8;
                if (a.out_dtype == AIR_KV_F32) {
                    float4 *dst = reinterpret_cast<float4 *>((float *)a.out + oi);
                    dst[0] = make_float4(acc[g][0] * inv, acc[g][1] * inv, acc[g][2] * inv, acc[g][3] * inv);
                    dst[1] = make_float4(acc[g][4] * inv, acc[g][5] * inv, acc[g][6] * inv, acc[g][7] * inv);
                } else {
                    uint32_t w[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        w[j] = (uint32_t)bf16_rne(acc[g][2 * j] * inv) |
                               ((uint32_t)bf16_rne(acc[g][2 * j + 1] * inv) << 16);
                    *reinterpret_cast<uint4 *>((uint16_t *)a.out + oi) = make_uint4(w[0], w[1], w[2], w[3]);
                }
            }
        }
    }
}

template <int DT, int G, int DP>
hipError_t launch_typed(const PrefillArgs &a, hipStream_t s) {
    // (row slot, kv head and head chunk, sequence)
    const int chunks = (a.group + G - 1) / G;
    const dim3 grid((unsigned)a.nz, (unsigned)(a.n_kv_heads * chunks), (unsigned)a.batch);
    hipLaunchKernelGGL((prefill_rows_kernel<DT, G, DP>), grid, dim3(kThreads), 0, s, a);
    return hipGetLastError();
}

// head_dim rounded up to 64, 128 or 256 lanes' worth of 8-element chunks
template <int DT, int G>
hipError_t launch_d(const PrefillArgs &a, hipStream_t s) {
    if (a.head_dim <= 64) return launch_typed<DT, G, 64>(a, s);
    if (a.head_dim <= 128) return launch_typed<DT, G, 128>(a, s);
    return launch_typed<DT, G, 256>(a, s);
}

// Heads per workgroup: the group rounded up to a power of two, at most 8 (4 up to
// head_dim 128, where larger groups only come here past 2^31 columns).
template <int DT>
hipError_t launch_g(const PrefillArgs &a, hipStream_t s) {
    if (a.group == 1) return launch_d<DT, 1>(a, s);
    if (a.group == 2) return launch_d<DT, 2>(a, s);
    if (a.group <= 4 || a.head_dim <= 128) return launch_d<DT, 4>(a, s);
    return launch_typed<DT, 8, 256>(a, s);
}

}  // namespace

hipError_t launch_prefill_rows(PrefillArgs a, int dtype, int32_t max_q_len, hipStream_t s) {
    // row slots per sequence: one per query row up to max_q_len (longer
    // chunks stride over them)
    a.nz = max_q_len < 1 ? 1 : (max_q_len > 65535 ? 65535 : max_q_len);
    switch (dtype) {
    case AIR_KV_F32: return launch_g<AIR_KV_F32>(a, s);
    case AIR_KV_BF16: return launch_g<AIR_KV_BF16>(a, s);
    case AIR_KV_INT8: return launch_g<AIR_KV_INT8>(a, s);
    default: return launch_g<AIR_KV_FP8>(a, s);
    }
}

}  // namespace airkv
