// Paged decode attention at f32 precision on the matrix cores: the pools and
// launches paged_decode_mfma.hip does not take -- f32 pages (the reference's
// own cache dtype), head_dim other than 128, scale groups below 32 and GQA
// groups above 16 (16 query heads of a kv head at a time; the reference's head
// map takes any group, src/chunked_attn.rs:65-72).
//
// The work division is paged_decode_mfma.hip's: equal slices of the batch's
// 16-token tiles, merged by log-sum-exp (src/flash_decode.rs:114-142).  A slice
// has one wave, or past 128 elements of head_dim the four of a workgroup, each
// with a quarter of the columns; they add their shares of a tile's scores
// through LDS.
//
// Per 16-token tile: v_mfma_f32_16x16x4_f32 takes one element per lane and
// operand, and the contraction order is free, so both operands come straight
// from wide page loads.
//   S = K . Q^T   lane (row r16 = lane % 16, g4 = lane / 16) holds 8 elements
//                 of token r16 per 32 of head_dim (key_elem below); product
//                 (m, e) contracts the four lanes' e-th ones.  bf16 pages
//                 under bf16 queries, and 1-byte codes (exact in bf16) whose
//                 scale holds for 32 elements, take v_mfma_f32_16x16x32_bf16
//                 instead, whose operand is those 8 elements: f32 queries in
//                 three bf16 parts (24 bits from 2^-110 on), the scale on each
//                 32 elements' sum.  Where rows are whole
//                 128-byte lines a load instruction reads eight of them, and a
//                 transpose of one lane bit with the load index (DPP) gives
//                 the lanes their elements; other rows are read directly, half
//                 a line of each per instruction.
//   O^T += V^T . P^T   step i contracts tokens 4 g4 + i, which is where the S
//                 product leaves P (lane: head r16, tokens 4 g4 + 0..3): the
//                 lane's elements of token 4 g4 + i are the other operand,
//                 with head_dim dealt out in pieces of up to 16 bytes.
// Every product is an f32 fused multiply-add (exact for bf16 operands); the
// scores run in eight chains and a tile's P.V starts from zero, so the running
// sums are rounded once per tile.  The values' 1-byte codes, and the keys' under
// f32 products, are dequantized (code * scale, one rounding) in registers.
//
// The decode step's new token (k_new / v_new) is written to its page by the
// wave that owns its sequence's last tile, just before it loads that tile:
// one launch, the same bytes as air_kv_append's.
//
// Bound by the page loads where the matrix cores keep up (f32 pages, bf16
// pages under bf16 queries), by the f32 products and the widening on 1-byte
// pages.  48 sequences of 256 to 4096 tokens, 32 heads over 8: bf16 pages of 64
// 49 us, 4.7 TB/s, 41 of them the slices' (180 us on the vector kernel this
// replaced, four launches); f32 pages of 64 88 us, 5.2 TB/s (204); 64 sequences
// of 256 to 8192 over int8 pages of 64 110 us, 3.2 TB/s (449).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "../host/status.hpp"
#include "../pool.hpp"
#include "bf16_parts.hpp"
#include "codecs.hpp"
#include "decode_common.hpp"
#include "decode_slices.hpp"
#include "page_io.hpp"

namespace airkv {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int kThreads = kSliceThreads;
constexpr int kWaves = kThreads / 64;
constexpr int kHeads = 16;                 // query heads of a kv head per wave
constexpr int kBufferWord3 = 0x00020000;   // raw buffer access
constexpr int kOutside = 1 << 30;          // a lane offset no page tile reaches: reads as zero
// Cache policy: loads that read whole lines are non-temporal (bf16 pages of 64,
// 48 sequences of 256 to 4096 tokens: 48.8 us, 50.2 with the keys cached, 54.5
// with both); key loads of half a line per instruction are cached.
constexpr int kLineAux = 2, kKeyAux = 0, kValueAux = 2;

constexpr int kF32 = AIR_KV_F32, kBf16 = AIR_KV_BF16, kInt8 = AIR_KV_INT8, kFp8 = AIR_KV_FP8;
template <int PT> constexpr bool kByte = PT == kInt8 || PT == kFp8;
template <int PT> constexpr int kElem = PT == kF32 ? 4 : PT == kBf16 ? 2 : 1;

// A lane's head_dim elements of a value row, D / 16 of them, in pieces of up
// to 16 bytes (8 elements): piece p holds SIZE elements from base + SIZE * (lane
// % 16), and 16 lanes' pieces are one contiguous run.
template <int D, int PT> struct Pieces {
    static constexpr int kMost = PT == kF32 ? 4 : 8, kEach = D / 16;
    static constexpr int kFull = kEach / kMost, kRest = kEach % kMost;
    static constexpr int N = kFull + ((kRest & 4) != 0) + ((kRest & 2) != 0);
    static constexpr int size(int p) { return p < kFull ? kMost : p == kFull && (kRest & 4) ? 4 : 2; }
    static constexpr int first(int p) { return p < kFull ? p * kMost : kFull * kMost + (p > kFull ? 4 : 0); }
    static_assert(kEach % 2 == 0, "head_dim in multiples of 32");
};

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void *p, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0, bytes, kBufferWord3);
}

template <int N> struct Int { static constexpr int value = N; };
// f(Int<0>) .. f(Int<N - 1>): loops whose index sizes types.
template <int N, int I = 0, class F> __device__ __forceinline__ void unrolled(F &&f) {
    if constexpr (I < N) {
        f(Int<I>{});
        unrolled<N, I + 1>(f);
    }
}

// BYTES at voff + soff of a page tile, as loaded (w: one word per 4 bytes).
template <int BYTES, int AUX>
__device__ __forceinline__ void load_words(__amdgpu_buffer_rsrc_t r, int voff, int soff, uint32_t *w) {
    if constexpr (BYTES == 32) {
        load_words<16, AUX>(r, voff, soff, w);
        load_words<16, AUX>(r, voff, soff + 16, w + 4);
    } else if constexpr (BYTES == 16) {
        const u32x4 x = __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, AUX);
#pragma unroll
        for (int i = 0; i < 4; ++i) w[i] = x[i];
    } else if constexpr (BYTES == 8) {
        const u32x2 x = __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, AUX);
        w[0] = x[0];
        w[1] = x[1];
    } else if constexpr (BYTES == 4) {
        w[0] = __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, AUX);
    } else {
        w[0] = __builtin_amdgcn_raw_buffer_load_b16(r, voff, soff, AUX);
    }
}

// Whether a word of fp8 codes holds 0xFF, which the hardware conversion below
// reads as NaN and the reference decoder as -480 (its encoder never gives it).
__device__ __forceinline__ uint32_t has_ff(uint32_t w) {
    return ((w & 0x7F7F7F7Fu) + 0x01010101u) & w & 0x80808080u;
}

// N loaded elements as f32 (FF: fp8 codes that may hold 0xFF).
template <int PT, int N, bool FF = false>
__device__ __forceinline__ void widen(const uint32_t *w, float s, float *x) {
#pragma clang fp contract(off)
    if constexpr (PT == kF32) {
#pragma unroll
        for (int j = 0; j < N; ++j) x[j] = __uint_as_float(w[j]);
    } else if constexpr (PT == kBf16) {
#pragma unroll
        for (int j = 0; j < N; ++j)
            x[j] = __uint_as_float((j & 1) ? w[j >> 1] & 0xFFFF0000u : w[j >> 1] << 16);
    } else if constexpr (PT == kFp8 && FF) {
#pragma unroll
        for (int j = 0; j < N; ++j) x[j] = fp8_decode((w[j >> 2] >> (8 * (j & 3))) & 0xFFu) * s;
    } else if constexpr (PT == kFp8) {
        // the hardware's OCP E4M3 conversion, after clearing the bytes with a
        // zero exponent field (+0 to the reference decoder), four at a time
#pragma unroll
        for (int i = 0; i < (N + 3) / 4; ++i) {
            const uint32_t nz = ((w[i] & 0x78787878u) + 0x78787878u) & 0x80808080u;
            const int c = (int)(w[i] & (nz | (nz - (nz >> 7))));
            const f32x2 lo = __builtin_amdgcn_cvt_pk_f32_fp8(c, false) * s;
            x[4 * i] = lo[0];
            x[4 * i + 1] = lo[1];
            if constexpr (N >= 4) {
                const f32x2 hi = __builtin_amdgcn_cvt_pk_f32_fp8(c, true) * s;
                x[4 * i + 2] = hi[0];
                x[4 * i + 3] = hi[1];
            }
        }
    } else {
#pragma unroll
        for (int j = 0; j < N; ++j) x[j] = (float)(int32_t)(int8_t)((w[j >> 2] >> (8 * (j & 3))) & 0xFFu) * s;
    }
}

// N (2, 4 or 8) consecutive outputs (bf16: the hardware's rounding to nearest even).
template <int N>
__device__ __forceinline__ void store_out(const DecodeArgs &a, int64_t i, const float *v) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    if (a.out_dtype == AIR_KV_F32) {
#pragma unroll
        for (int j = 0; j < N; j += 2) *reinterpret_cast<f32x2 *>((float *)a.out + i + j) = f32x2{v[j], v[j + 1]};
    } else {
#pragma unroll
        for (int j = 0; j < N; j += 2)
            *reinterpret_cast<uint32_t *>((uint16_t *)a.out + i + j) =
                __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{v[j], v[j + 1]}), bf16x2));
    }
}

// A workgroup barrier that orders LDS only (page loads stay in flight).
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Waves per SIMD an instantiation is built for and launched with.
template <int D, int PT, int QP> constexpr int waves_per_simd() {
    return PT == kF32                  ? (D <= 64 ? 3 : 2)
           : PT == kBf16 && QP == 1    ? (D <= 96 ? 4 : D <= 128 ? 3 : 2)
           : D <= 64  ? (PT == kBf16 ? 4 : 3)
           : D <= 96  ? 3
                      : (PT == kBf16 ? 3 : 2);
}

// D: a wave's columns.  QP: the scores' products, 0 f32 (the queries as f32), 1 bf16
// under bf16 queries, 3 bf16 under f32 queries in three parts.  TEAM: the
// workgroup's waves share a slice, D columns of head_dim each.
template <int D, int PT, int QP, bool TEAM>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(waves_per_simd<D, PT, QP>(), waves_per_simd<D, PT, QP>())))
void decode_f32_kernel(DecodeArgs a) {
    static_assert(QP == 0 || PT != kF32, "bf16 products take bf16 pages or codes");
    using P = Pieces<D, PT>;
    constexpr int EB = kElem<PT>, KM = D / 32;
    __shared__ int32_t s_pre[kMaxBatch + 2];
    __shared__ int32_t s_wsum[kWaves];
    __shared__ uint32_t s_long[kMaxBatch / 32];  // the step: sequences longer than their table append nothing
    tile_prefix(a, a.block_size, s_pre, s_wsum, s_long);
    const int B = a.batch;
    const int total = s_pre[B];
    const int chunk = a.seq_pieces ? 0 : shared_chunk(total, a.slices, a.simd_slices, s_pre[B + 1], a.max_splits);
    if (blockIdx.x == 0) {                     // for the merge kernel: prefix, then the chunk
        for (int i = threadIdx.x; i <= B; i += kThreads) a.prefix[i] = s_pre[i];
        if (threadIdx.x == 0) a.prefix[B + 1] = chunk;
    }
    __shared__ f32x4 s_part[TEAM ? 2 : 1][TEAM ? kWaves : 1][TEAM ? 64 : 1];   // a tile's scores by wave
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g4 = lane >> 4, r16 = lane & 15;
    const int G = a.group, d = a.head_dim;
    const int col0 = TEAM ? D * wave : 0, dw = d - col0;        // the wave's columns: the first D of dw (none: dw <= 0)
    // Consecutive waves (or teams) take consecutive kv heads of one slice
    // (neighbouring pages), then the slice's other head chunks.
    const int gw = TEAM ? (int)blockIdx.x : blockIdx.x * kWaves + wave;
    const int chunks = (G + kHeads - 1) / kHeads;
    const int kh = gw % a.n_kv_heads, rest = gw / a.n_kv_heads;
    const int hc = rest % chunks, w = rest / chunks;
    int lo, hi;                                // the slice's tiles
    if (a.seq_pieces) {
        const int b = w / a.seq_pieces;
        if (b >= B) return;
        const int step = piece_tiles(s_pre[b + 1] - s_pre[b], a.seq_pieces);
        lo = s_pre[b] + w % a.seq_pieces * step;
        hi = s_pre[b + 1] - lo < step ? s_pre[b + 1] : lo + step;
        if (lo >= hi) return;
    } else {
        if (w >= a.slices || (int64_t)w * chunk >= total) return;
        lo = w * chunk;
        hi = total - lo < chunk ? total : lo + chunk;
    }
    lo = __builtin_amdgcn_readfirstlane(lo);
    hi = __builtin_amdgcn_readfirstlane(hi);
    const int g0 = hc * kHeads, gn = G - g0 < kHeads ? G - g0 : kHeads;   // this wave's heads of the group
    const int64_t max_len = (int64_t)a.max_blocks * a.block_size;
    const int bs_log2 = __builtin_ctz((unsigned)a.block_size);
    const int sg_log2 = kByte<PT> ? __builtin_ctz((unsigned)a.scale_group) : 0;
    const int n_sc = kByte<PT> ? d >> sg_log2 : 0;

    // Lane k of a 64-tile window describes tile c0 + k: sequence, block id,
    // tile of the sequence, valid tokens.
    int32_t tbl = 0, seq_l = 0, j_l = 0, nv_l = 0;
    uint64_t first_m = 0, last_m = 0, new_m = 0;   // tile starts / ends a piece / holds the step's new token
    auto load_window = [&](int c0) {
        const int t = c0 + lane < hi ? c0 + lane : hi - 1;
        const int bq = seq_of_tile(s_pre, B, t);
        const int j = t - s_pre[bq];
        const int64_t len = clamp_len(a.lens[bq], max_len);
        tbl = a.tables[(int64_t)bq * a.max_blocks + ((16 * j) >> bs_log2)];
        seq_l = bq;
        j_l = j;
        const int64_t left = len - 16 * (int64_t)j;
        nv_l = left < 16 ? (int)left : 16;
        const bool valid = c0 + lane < hi;
        first_m = __ballot(valid && (t == lo || j == 0));
        last_m = __ballot(valid && (t + 1 == hi || t + 1 == s_pre[bq + 1]));
        new_m = a.k_new ? __ballot(valid && t + 1 == s_pre[bq + 1] && !((s_long[bq >> 5] >> (bq & 31)) & 1)) : 0;
    };

    // The lane's elements of 32: 8 g4 .. + 8, or for f32 pages read by lines, as
    // their two 16-byte loads come, 4 g4 .. + 4 and 16 + 4 g4 .. + 4.
    auto key_elem = [&](int half) { return PT == kF32 ? 16 * half + 4 * g4 : 8 * g4 + 4 * half; };
    // ---- queries (head r16), the same elements; heads past the chunk and
    // columns past head_dim read zeros outside the descriptor
    u32x4 qb[QP ? QP : 1][QP ? KM : 1];
    float qf[QP ? 1 : KM][8];
    auto load_q = [&](int bq) __attribute__((always_inline)) {
        const int qbytes = a.q_dtype == AIR_KV_F32 ? 4 : 2;
        const int64_t row = (int64_t)bq * a.n_q_heads + kh * G + g0;
        const __amdgpu_buffer_rsrc_t rq = rsrc((const char *)a.q + row * d * qbytes, gn * d * qbytes);
#pragma unroll
        for (int m = 0; m < KM; ++m) {
            const int off = (r16 * d + col0 + 32 * m) * qbytes;
            if constexpr (QP == 1) {
                qb[0][m] = __builtin_amdgcn_raw_buffer_load_b128(rq, 32 * m < dw ? off + 16 * g4 : kOutside, 0, 0);
            } else if constexpr (QP == 3) {
                uint32_t x[8];
                load_words<32, 0>(rq, 32 * m < dw ? off + 32 * g4 : kOutside, 0, x);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    uint32_t h, mid, l;
                    split3(__uint_as_float(x[2 * j]), __uint_as_float(x[2 * j + 1]), h, mid, l);
                    qb[0][m][j] = h;
                    qb[1][m][j] = mid;
                    qb[2][m][j] = l;
                }
            } else {
#pragma unroll
                for (int half = 0; half < 2; ++half) {
                    const int at = 32 * m < dw ? off + key_elem(half) * qbytes : kOutside;
                    uint32_t x[4];
                    if (a.q_dtype == AIR_KV_F32) {
                        load_words<16, 0>(rq, at, 0, x);
                        widen<kF32, 4>(x, 1.0f, &qf[m][4 * half]);
                    } else {
                        load_words<8, 0>(rq, at, 0, x);
                        widen<kBf16, 4>(x, 1.0f, &qf[m][4 * half]);
                    }
                }
            }
        }
    };

    f32x4 acc[P::N][P::kMost];               // O^T: piece p, element j: rows i = piece lane 4 g4 + i, column head r16
    float m_run = -INFINITY, l_run = 0.0f;

    // Lane offsets in a tile: key chunk m of row r16, value piece p of row
    // 4 g4 (step i adds i rows), and their scales.
    // Whole-line key loads: load h of a 128-byte line column reads, in lane
    // l, row 8 h + l % 8, 16 bytes at 64 bit3(l) + 32 bit5(l) + 16 bit4(l).
    constexpr bool LINES = !kByte<PT> && D * EB % 128 == 0;
    const bool lines = LINES && d * EB % 128 == 0;
    const int k_off = col0 * EB + (lines ? (lane & 7) * d * EB + 64 * ((lane >> 3) & 1) + 32 * (lane >> 5) + 16 * ((lane >> 4) & 1)
                                         : (r16 * d + 8 * g4) * EB);
    const int v_off = (4 * g4 * d + col0) * EB;
    uint32_t kw[KM][8 * EB / 4], vw[4][P::N][P::kMost * EB / 4 > 0 ? P::kMost * EB / 4 : 1];
    float ksc[kByte<PT> ? KM : 1][QP ? 4 : 1], vsc[kByte<PT> ? 4 : 1][kByte<PT> ? P::N : 1];

    __amdgpu_buffer_rsrc_t rv, rvs;
    auto load_values = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            unrolled<P::N>([&](auto pc) {
                constexpr int p = decltype(pc)::value, SZ = P::size(p), base = 16 * P::first(p);
                const int voff = base + SZ * r16 < dw ? v_off + SZ * r16 * EB : kOutside;
                load_words<SZ * EB, kValueAux>(rv, voff, (i * d + base) * EB, vw[i][p]);
            });
        if constexpr (kByte<PT>) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                unrolled<P::N>([&](auto pc) {
                    constexpr int p = decltype(pc)::value;
                    const int at = 16 * P::first(p) + P::size(p) * r16;
                    vsc[i][p] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
                        rvs, at < dw ? (4 * g4 * n_sc + ((col0 + at) >> sg_log2)) * 4 : kOutside, i * n_sc * 4, 0));
                });
        }
    };
    auto load_tile = [&](int idx) -> bool {
        int32_t blk = __builtin_amdgcn_readlane(tbl, idx);
        const int j = __builtin_amdgcn_readlane(j_l, idx);
        const bool ok = blk >= 0 && blk < a.num_blocks;
        blk = ok ? blk : 0;
        const int64_t row0 = ((int64_t)blk * a.n_kv_heads + kh) * a.block_size + ((16 * j) & (a.block_size - 1));
        if (ok && ((new_m >> idx) & 1)) {
            // the step's new token: row nv - 1 of this tile, lanes 0 .. d/8 - 1
            // its key, the next d/8 its value; in the page before the tile
            // loads (the waves of a team and of a group's head chunks each write
            // the same bytes, so none depends on another's)
            const int bq = __builtin_amdgcn_readlane(seq_l, idx);
            const int64_t row = row0 + __builtin_amdgcn_readlane(nv_l, idx) - 1;
            const int per = d >> 3, c = lane < per ? lane : lane - per;
            const bool val = lane >= per, live = lane < 2 * per;
            float x[8];
            const float *src = (val ? a.v_new : a.k_new) + ((int64_t)bq * a.n_kv_heads + kh) * d + 8 * (live ? c : 0);
            const f32x4 x0 = *reinterpret_cast<const f32x4 *>(src), x1 = *reinterpret_cast<const f32x4 *>(src + 4);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                x[i] = x0[i];
                x[4 + i] = x1[i];
            }
            void *pg = const_cast<void *>(val ? a.v_pages : a.k_pages);
            float *sc = const_cast<float *>(val ? a.v_scales : a.k_scales);
            const int lpg = kByte<PT> ? a.scale_group >> 3 : 1;
            const int64_t elem = row * d + 8 * c, sidx = row * n_sc + ((8 * c) >> sg_log2);
            store_row_chunk<PT>(x, pg, sc, elem, sidx, c % lpg == 0, lpg, live);
            __builtin_amdgcn_s_waitcnt(0);               // written before the loads below are issued
            asm volatile("" ::: "memory");
        }
        // rows past the sequence, and a block outside the pool, read as zeros
        // without a memory access
        const int nv = ok ? __builtin_amdgcn_readlane(nv_l, idx) : 0;
        const __amdgpu_buffer_rsrc_t rk = rsrc((const char *)a.k_pages + row0 * d * EB, nv * d * EB);
        rv = rsrc((const char *)a.v_pages + row0 * d * EB, nv * d * EB);
        if (lines) {
            // line column c: words 8 c .. + 8 of kw, one 16-byte load each half
#pragma unroll
            for (int c = 0; c < KM * 8 * EB / 32; ++c)
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    load_words<16, kLineAux>(rk, 128 * c < dw * EB ? k_off : kOutside, 128 * c + 8 * h * d * EB,
                                             &kw[0][0] + 8 * c + 4 * h);
        } else {
#pragma unroll
            for (int m = 0; m < KM; ++m) {
                load_words<8 * EB, kKeyAux>(rk, 32 * m < dw ? k_off : kOutside, 32 * m * EB, kw[m]);
            }
        }
        if constexpr (kByte<PT>) {
            const __amdgpu_buffer_rsrc_t rks = rsrc(a.k_scales + row0 * n_sc, nv * n_sc * 4);
            rvs = rsrc(a.v_scales + row0 * n_sc, nv * n_sc * 4);
            // of the lane's own row, or (QP) of the four rows of its scores
#pragma unroll
            for (int m = 0; m < KM; ++m)
#pragma unroll
                for (int i = 0; i < (QP ? 4 : 1); ++i)
                    ksc[m][i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
                        rks, 32 * m < dw ? ((QP ? 4 * g4 : r16) * n_sc + ((col0 + 32 * m + (QP ? 0 : 8 * g4)) >> sg_log2)) * 4 : kOutside,
                        i * n_sc * 4, 0));
        }
        load_values();
        return ok;
    };

    // The piece of sequence bq held by this wave ends: write it out.
    auto emit = [&](int bq) __attribute__((always_inline)) {
        const float l = sum_x32(sum_x16(l_run));
        const bool starts = s_pre[bq] >= lo;
        if (r16 >= gn) return;
        const bool whole = starts && s_pre[bq + 1] <= hi;   // the whole sequence: final output
        const bool none = whole && !(l > 0.0f);  // no sum, every key at -inf: zeros, as the merge gives
        const float inv = whole ? 1.0f / l : 1.0f;
        const int64_t orow = ((int64_t)bq * a.n_q_heads + kh * G + g0 + r16) * d + col0;
        const int64_t prow = ((int64_t)kh * a.slots + (a.seq_pieces ? w : part_row(w, bq, starts))) * G + g0 + r16;
        unrolled<P::N>([&](auto pc) {
            constexpr int p = decltype(pc)::value, SZ = P::size(p);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int at = 16 * P::first(p) + SZ * (4 * g4 + i);
                if (at >= dw) continue;
                float v[SZ];
#pragma unroll
                for (int j = 0; j < SZ; ++j) v[j] = none ? 0.0f : acc[p][j][i] * inv;
                if (whole) {
                    store_out<SZ>(a, orow + at, v);
                } else {
#pragma unroll
                    for (int j = 0; j < SZ; j += 2)
                        *reinterpret_cast<f32x2 *>(a.part_o + prow * d + col0 + at + j) = f32x2{v[j], v[j + 1]};
                }
            }
        });
        if (!whole && g4 == 0 && col0 == 0) {
            a.part_ml[prow * 2] = m_run;
            a.part_ml[prow * 2 + 1] = l;
        }
    };

    auto compute_tile = [&](auto ffc, int k, int idx, bool ok) __attribute__((always_inline)) {
        constexpr bool FF = decltype(ffc)::value != 0;
        const int bq = __builtin_amdgcn_readlane(seq_l, idx);
        if ((first_m >> idx) & 1) {              // a new sequence starts in this slice
            if (k != lo) load_q(bq);
            m_run = -INFINITY;
            l_run = 0.0f;
#pragma unroll
            for (int p = 0; p < P::N; ++p)
#pragma unroll
                for (int j = 0; j < P::kMost; ++j) acc[p][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        }
        // a table entry outside the pool is counted and its tile masked out
        if (!ok && lane == 0 && hc == 0 && col0 == 0) atomicAdd(a.errors, 1ull);
        const int nv = ok ? __builtin_amdgcn_readlane(nv_l, idx) : 0;
        if constexpr (LINES) {
            if (lines) {
#pragma unroll
                for (int c = 0; c < KM * 8 * EB / 32; ++c) {
                    uint32_t *x = &kw[0][0] + 8 * c;
                    u32x4 x0 = {x[0], x[1], x[2], x[3]}, x1 = {x[4], x[5], x[6], x[7]};
                    swap_lane_bit3(x0, x1);
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        x[j] = x0[j];
                        x[4 + j] = x1[j];
                    }
                }
            }
        }
        // S: lane holds tokens 4 g4 + i of head r16; every product starts from
        // zero and the partial sums are added pairwise
        const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
        f32x4 part[KM];
#pragma unroll
        for (int m = 0; m < KM; ++m) {
            if constexpr (QP) {
                u32x4 ka;
                if constexpr (PT == kBf16) {
                    ka = u32x4{kw[m][0], kw[m][1], kw[m][2], kw[m][3]};
                } else {
                    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
                    float x[8];
                    widen<PT, 8, FF>(kw[m], 1.0f, x);
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        ka[j] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{x[2 * j], x[2 * j + 1]}), bf16x2));
                }
                part[m] = zero;
#pragma unroll
                for (int p = QP - 1; p >= 0; --p)        // the least part first
                    part[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        __builtin_bit_cast(bf16x8, ka), __builtin_bit_cast(bf16x8, qb[p][m]), part[m], 0, 0, 0);
                if constexpr (kByte<PT>)
#pragma unroll
                    for (int i = 0; i < 4; ++i) part[m][i] *= ksc[m][QP ? i : 0];
            } else {
                float x[8];
                widen<PT, 8, FF>(kw[m], kByte<PT> ? ksc[kByte<PT> ? m : 0][0] : 1.0f, x);
                f32x4 c[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) c[e] = mfma4(x[e], qf[m][e], zero);
                part[m] = ((c[0] + c[1]) + (c[2] + c[3])) + ((c[4] + c[5]) + (c[6] + c[7]));
                __builtin_amdgcn_sched_barrier(0);       // one chunk's elements widened at a time
            }
        }
#pragma unroll
        for (int st = 1; st < KM; st <<= 1)
#pragma unroll
            for (int m = 0; m + st < KM; m += 2 * st) part[m] += part[m + st];
        f32x4 s = part[0];
        if constexpr (TEAM) {
            // the columns' shares, added in one order by every wave.  Two
            // buffers, one barrier a tile: a wave writes a buffer again only
            // past the barrier of the tile between, which it reached after
            // reading this one, as all of them did.
            f32x4 (*sp)[64] = s_part[k & 1];
            sp[wave][lane] = s;
            lds_barrier();
            s = (sp[0][lane] + sp[1][lane]) + (sp[2][lane] + sp[3][lane]);
        }
        float sc[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) sc[i] = s[i] * a.scale_log2;
        const bool full = nv == 16;              // uniform: only a sequence's last tile is partial
        if (!full) {
#pragma unroll
            for (int i = 0; i < 4; ++i) sc[i] = 4 * g4 + i < nv ? sc[i] : -INFINITY;
        }
        float mt = fmaxf(fmaxf(sc[0], sc[1]), fmaxf(sc[2], sc[3]));
        mt = max_x32(max_x16(mt));
        // (no slack here: probabilities above 1 would overflow on values near
        // the largest f32)
        if (__ballot(mt > m_run) != 0ull) {
            const float m_new = fmaxf(m_run, mt);
            const float alpha = (m_run == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f(m_run - m_new);
            l_run *= alpha;
#pragma unroll
            for (int p = 0; p < P::N; ++p)
#pragma unroll
                for (int j = 0; j < P::kMost; ++j) acc[p][j] *= alpha;
            m_run = m_new;
        }
        float pr[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) pr[i] = (sc[i] == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f(sc[i] - m_run);
        l_run += (pr[0] + pr[1]) + (pr[2] + pr[3]);
        unrolled<P::N>([&](auto pc) {
            constexpr int p = decltype(pc)::value, SZ = P::size(p);
            float x[4][SZ];
#pragma unroll
            for (int i = 0; i < 4; ++i)
                widen<PT, SZ, FF>(vw[i][p], kByte<PT> ? vsc[kByte<PT> ? i : 0][kByte<PT> ? p : 0] : 1.0f, x[i]);
#pragma unroll
            for (int j = 0; j < SZ; ++j) {
                const f32x4 o0 = mfma4(x[1][j], pr[1], mfma4(x[0][j], pr[0], zero));
                const f32x4 o1 = mfma4(x[3][j], pr[3], mfma4(x[2][j], pr[2], zero));
                acc[p][j] += o0 + o1;
            }
            if constexpr (kByte<PT>) __builtin_amdgcn_sched_barrier(0);
        });
        if (__builtin_expect((last_m >> idx) & 1, 0)) emit(bq);
    };

    for (int c0 = lo; c0 < hi; c0 += 64) {
        load_window(c0);
        if (c0 == lo) load_q(__builtin_amdgcn_readlane(seq_l, 0));
        const int n = hi - c0 < 64 ? hi - c0 : 64;
        for (int i = 0; i < n; ++i) {
            const bool ok = load_tile(i);
            if constexpr (PT == kFp8) {
                uint32_t ff = 0;
#pragma unroll
                for (int m = 0; m < KM; ++m) ff |= has_ff(kw[m][0]) | has_ff(kw[m][1]);
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    unrolled<P::N>([&](auto pc) {
                        constexpr int p = decltype(pc)::value;
                        ff |= has_ff(vw[j][p][0]);
                        if constexpr (P::size(p) == 8) ff |= has_ff(vw[j][p][1]);
                    });
                if (__builtin_expect(__ballot(ff != 0) != 0, 0)) {
                    compute_tile(Int<1>{}, c0 + i, i, ok);
                    continue;
                }
            }
            compute_tile(Int<0>{}, c0 + i, i, ok);
        }
    }
}

// Log-sum-exp merge of a (sequence, query head)'s pieces by one wave: groups
// of L = DP / 4 lanes (DP: head_dim rounded up to 64, 128 or 256) hold four
// columns a lane and fold every 64 / L-th piece, kBatch of them per memory
// round trip, then the groups are folded across the wave.  Also zeros for an
// empty sequence, and the count of lengths outside the table.
template <int DP>
__global__ __launch_bounds__(kThreads) void decode_f32_merge_kernel(DecodeArgs a) {
    constexpr int L = DP / 4, NG = 64 / L, kBatch = 4;
    const int b = blockIdx.x, kh = blockIdx.y, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int G = a.group, d = a.head_dim, h = blockIdx.z * kWaves + wave;
    const int64_t max_len = (int64_t)a.max_blocks * a.block_size;
    const int p0 = a.prefix[b], p1 = a.prefix[b + 1], chunk = a.prefix[a.batch + 1];
    const int len = a.lens[b];
    if (threadIdx.x == 0 && kh == 0 && blockIdx.z == 0 && (len < 0 || len > max_len)) atomicAdd(a.errors, 1ull);
    if (h >= G) return;
    const int col = lane % L * 4, grp = lane / L;
    const bool mine = col < d;
    const int64_t oi = ((int64_t)b * a.n_q_heads + kh * G + h) * d + col;
    float o[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (p0 != p1) {
        const int step = a.seq_pieces ? piece_tiles(p1 - p0, a.seq_pieces) : chunk;
        const int w0 = a.seq_pieces ? 0 : p0 / step;
        const int n = a.seq_pieces ? (p1 - p0 + step - 1) / step : (p1 - 1) / step - w0 + 1;
        if (n == 1) return;                              // written by its slice
        float m = -INFINITY, l = 0.0f;
        auto fold = [&](float pm, float pl, f32x4 pv) {
            if (pm == -INFINITY) return;
            const float m_new = fmaxf(m, pm);
            const float sa = __builtin_amdgcn_exp2f(m - m_new), sb = __builtin_amdgcn_exp2f(pm - m_new);
            l = l * sa + pl * sb;
#pragma unroll
            for (int i = 0; i < 4; ++i) o[i] = o[i] * sa + pv[i] * sb;
            m = m_new;
        };
        for (int q = 0; q < n; q += NG * kBatch) {
            float pm[kBatch], pl[kBatch];
            f32x4 pv[kBatch];
#pragma unroll
            for (int i = 0; i < kBatch; ++i) {
                const int p = q + NG * i + grp;
                const int w = w0 + (p < n ? p : 0);
                const int64_t row =
                    ((int64_t)kh * a.slots + (a.seq_pieces ? b * a.seq_pieces + w : part_row(w, b, w == w0))) * G + h;
                pm[i] = p < n ? a.part_ml[row * 2] : -INFINITY;
                pl[i] = a.part_ml[row * 2 + 1];
                pv[i] = *reinterpret_cast<const f32x4 *>(a.part_o + row * d + (mine ? col : 0));
            }
#pragma unroll
            for (int i = 0; i < kBatch; ++i) fold(pm[i], pl[i], pv[i]);
        }
#pragma unroll
        for (int x = L; x < 64; x <<= 1) {
            const float pm = __shfl_xor(m, x), pl = __shfl_xor(l, x);
            const f32x4 pv = {__shfl_xor(o[0], x), __shfl_xor(o[1], x), __shfl_xor(o[2], x), __shfl_xor(o[3], x)};
            fold(pm, pl, pv);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = l > 0.0f ? o[i] / l : 0.0f;   // (no sum, every key at -inf: zeros)
    }
    if (grp == 0 && mine) store_out<4>(a, oi, o);
}

template <int D, int PT, int QP, bool TEAM>
hipError_t launch_one(const DecodeArgs &a, hipStream_t s) {
    const int chunks = (a.group + kHeads - 1) / kHeads;
    const int64_t units = (int64_t)a.n_kv_heads * chunks * a.slices, per = TEAM ? 1 : kWaves;
    hipLaunchKernelGGL((decode_f32_kernel<D, PT, QP, TEAM>), dim3((unsigned)((units + per - 1) / per)), dim3(kThreads),
                       0, s, a);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const dim3 grid((unsigned)a.batch, (unsigned)a.n_kv_heads, (unsigned)((a.group + kWaves - 1) / kWaves));
    if constexpr (TEAM || D > 128) hipLaunchKernelGGL(decode_f32_merge_kernel<256>, grid, dim3(kThreads), 0, s, a);
    else if constexpr (D <= 64) hipLaunchKernelGGL(decode_f32_merge_kernel<64>, grid, dim3(kThreads), 0, s, a);
    else hipLaunchKernelGGL(decode_f32_merge_kernel<128>, grid, dim3(kThreads), 0, s, a);
    return hipGetLastError();
}

template <int D, bool TEAM>
hipError_t launch_d(const DecodeArgs &a, int dtype, hipStream_t s) {
    const bool q_bf16 = a.q_dtype == AIR_KV_BF16;
    if (dtype == AIR_KV_F32) return launch_one<D, kF32, 0, TEAM>(a, s);
    if (dtype == AIR_KV_BF16) return q_bf16 ? launch_one<D, kBf16, 1, TEAM>(a, s) : launch_one<D, kBf16, 0, TEAM>(a, s);
    // Codes take f32 products where a scale holds for fewer than 32 elements, and
    // fp8 codes past 64 columns under f32 queries (their two copies of a tile's
    // arithmetic spill with three parts: 100 sequences of 400 to 800, 8 kv heads,
    // pages of 96 70 us, 76 with them).  Elsewhere bf16 products are faster: 115
    // of 4245 to 8491, 4 heads over 4, int8 pages of 64 130 us, 184 with f32
    // products, 167 on the vector kernel before them.
    const bool wide = a.scale_group >= 32;
    if (dtype == AIR_KV_INT8)
        return !wide    ? launch_one<D, kInt8, 0, TEAM>(a, s)
               : q_bf16 ? launch_one<D, kInt8, 1, TEAM>(a, s)
                        : launch_one<D, kInt8, 3, TEAM>(a, s);
    if (wide && q_bf16) return launch_one<D, kFp8, 1, TEAM>(a, s);
    if constexpr (D <= 64)
        if (wide) return launch_one<D, kFp8, 3, TEAM>(a, s);
    return launch_one<D, kFp8, 0, TEAM>(a, s);
}

// Past 128 elements a wave that holds a whole tile runs alone on its SIMD with
// nothing to overlap, so a workgroup's four waves share the tile, 64 columns
// each (88 sequences of 114 tokens, 8 heads over 4, f32 pages of 256: 25.9 us, 37.2
// with a wave alone, 30.0 on the vector kernel before it).  Two waves of 96 columns
// for up to 192 elements were 2 to 10% slower.
constexpr int kTeamColumns = 64;
bool team(int d) { return d > 128; }

// Two waves of bf16 products fit a SIMD with a whole tile each, and need no
// barrier: under bf16 queries a launch over bf16 pages takes them where they have
// 20 tiles a SIMD to walk and the partitions alone are as many (16 sequences of
// 6000 to 12000, 16 heads over 8, pages of 160: 148 us, 188 shared by four; 5 of 2459
// to 19678, 16 over 4, pages of 256, below both: 70 and 46).  The table's width
// stands for the lengths.
bool lone_bf16(const air_kv_pool &p, int64_t per_slice, int64_t batch, int64_t tiles, int64_t max_splits) {
    return team(p.desc.head_dim) && p.desc.dtype == AIR_KV_BF16 && batch * tiles * per_slice >= (int64_t)80 * p.cus &&
           batch * std::min(tiles, max_splits) * per_slice >= (int64_t)8 * p.cus;
}

template <int D> int waves_of(int dtype, bool q_bf16) {
    return dtype == AIR_KV_F32    ? waves_per_simd<D, kF32, 0>()
           : dtype == AIR_KV_INT8 ? waves_per_simd<D, kInt8, 0>()
           : dtype == AIR_KV_FP8  ? waves_per_simd<D, kFp8, 0>()
           : q_bf16               ? waves_per_simd<D, kBf16, 1>()
                                  : waves_per_simd<D, kBf16, 0>();
}

}  // namespace

static_assert(kWsBytes <= (size_t)AIR_KV_NOALLOC_SCRATCH_BYTES, "air_paged_decode_noalloc holds the plan's workspace");

int plan_decode_f32(const air_kv_pool &p, int32_t n_q_heads, int32_t batch, int32_t max_blocks,
                    int32_t max_splits, DecodePlan *plan) {
    const int nkv = p.desc.n_kv_heads, d = p.desc.head_dim, dt = p.desc.dtype;
    const int64_t per_slice = (int64_t)nkv * ((n_q_heads / nkv + kHeads - 1) / kHeads);
    const int64_t tiles = std::min<int64_t>(((int64_t)max_blocks * p.desc.block_size + 15) / 16, INT32_MAX);
    plan->lone = lone_bf16(p, per_slice, batch, tiles, max_splits);
    auto waves = [&](bool q_bf16) {
        if (q_bf16 && plan->lone) return (int64_t)p.cus * 4 * waves_per_simd<256, kBf16, 1>();
        const int wps = d <= 64    ? waves_of<64>(dt, q_bf16)
                        : d <= 96  ? waves_of<96>(dt, q_bf16)
                        : !team(d) ? waves_of<128>(dt, q_bf16)
                                   : waves_of<kTeamColumns>(dt, q_bf16);
        return (int64_t)p.cus * (team(d) ? 1 : 4) * wps;
    };
    const DecodeF32Plan pl = plan_f32(n_q_heads, per_slice, d, p.desc.block_size, batch, max_blocks, max_splits,
                                      waves(true), waves(false));
    plan->mfma = false;
    plan->dtype = dt;
    plan->slices = (int32_t)pl.slices;
    plan->slices_qf32 = (int32_t)pl.slices_qf32;
    plan->slices_append = 0;
    plan->seq_pieces = (int32_t)pl.seq_pieces;
    plan->batch_per_launch = (int32_t)pl.batch;
    plan->slots = (int32_t)pl.slots;
    plan->ws_bytes = pl.ws_bytes;
    return AIR_KV_OK;
}

hipError_t launch_decode_f32(const DecodeArgs &base, const DecodePlan &plan, void *workspace, hipStream_t s) {
    const int d = base.head_dim;
    for (int32_t b0 = 0; b0 < base.batch; b0 += plan.batch_per_launch) {
        DecodeArgs a = base;
        a.batch = std::min(base.batch - b0, plan.batch_per_launch);
        a.slices = base.q_dtype == AIR_KV_F32 ? plan.slices_qf32 : plan.slices;
        a.slots = plan.slots;
        const bool lone = plan.lone && base.q_dtype == AIR_KV_BF16;
        a.simd_slices = team(d) && !lone ? (base.simd_slices + kWaves - 1) / kWaves : base.simd_slices;
        const int64_t q_row = (int64_t)b0 * a.n_q_heads * d;
        a.q = (const char *)base.q + q_row * (base.q_dtype == AIR_KV_F32 ? 4 : 2);
        a.out = (char *)base.out + q_row * (base.out_dtype == AIR_KV_F32 ? 4 : 2);
        a.tables = base.tables + (int64_t)b0 * a.max_blocks;
        a.lens = base.lens + b0;
        if (base.k_new) {
            const int64_t kv_row = (int64_t)b0 * a.n_kv_heads * d;
            a.k_new = base.k_new + kv_row;
            a.v_new = base.v_new + kv_row;
        }
        char *ws = (char *)workspace;
        const size_t rows = (size_t)a.n_q_heads * plan.slots;
        a.prefix = (int32_t *)ws;
        ws += decode_align256((size_t)(plan.batch_per_launch + 2) * 4);
        a.part_ml = (float *)ws;
        ws += decode_align256(rows * 2 * 4);
        a.part_o = (float *)ws;
        const hipError_t e = d <= 64    ? launch_d<64, false>(a, plan.dtype, s)
                             : d <= 96  ? launch_d<96, false>(a, plan.dtype, s)
                             : !team(d) ? launch_d<128, false>(a, plan.dtype, s)
                             : lone     ? launch_one<256, kBf16, 1, false>(a, s)
                                        : launch_d<kTeamColumns, true>(a, plan.dtype, s);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace airkv
