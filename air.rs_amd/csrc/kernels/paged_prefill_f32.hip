// Paged prefill attention (chunked, causal) at f32 precision on the matrix
// cores: the pools paged_prefill.hip does not take -- f32 pages (the
// reference's own cache dtype) and head_dim other than 128.
//
// Semantics are paged_prefill.hip's (blockwise_attention_head with q_offset =
// seq_len - q_len, src/chunked_attn.rs:114-213, over paged storage).  What
// differs is the arithmetic: queries, keys, probabilities, values and sums
// keep their 24 bits between 2^-110 and the largest f32.  An f32 operand enters
// v_mfma_f32_32x32x16_bf16 as three bf16 parts, each the rounding of what the
// parts before it leave (8 bits a part, the exponent range of f32), and a product
// of two such operands is the six part products down to 2^-16; bf16 queries and
// bf16 pages are one part as they are.  The matrix cores run those six at 2.7
// times the rate of their own f32 products.  1-byte codes are dequantized (code *
// scale, one rounding) as they are staged.  Below 2^-110 the parts under 2^-126
// are lost: f32 values of 1e-37 keep 13 bits.  (Computing their columns again as
// below, found by the least query element and output, cost every small launch
// 1.5 to 4%.)
//
// Rounding of the sums: the part products below the leading ones are added
// first (in the scores, in an accumulator of their own), and a tile's P.V
// starts from zero and joins the running output with one addition, so the
// running sum is rounded once per tile.
//
// Work: the (query row, head of the GQA group) pairs of one (sequence, kv
// head) are numbered row-major, and a workgroup of four waves takes 128 / NK
// consecutive ones: 32 to a wave, the columns of its products, and the waves
// of a column set share its keys NK ways.  A short chunk's rows times its
// group so fill whole waves, and every K / V tile staged in LDS serves all of
// them.  NK > 1 is for launches of few workgroups (launch_nk): the waves of a
// set walk every NK-th 32 keys and are combined by log-sum-exp in LDS (the
// combination of src/flash_decode.rs:114-142).
//
// Tiles of KT keys are staged row-major in LDS, in two buffers where they fit
// (one barrier per tile), with the loads of the next tile in flight in
// registers while one is computed.  The row pitches keep the operand reads
// free of bank conflicts.
//
// A column whose result is not finite is computed again by one wave with
// plain f32 arithmetic over its own keys only (slow_column): the products
// above also read the keys behind the causal mask, where a non-finite value
// times a zero probability would give NaN, and the parts of an infinity are
// not finite numbers.
//
// Bound by vector issue (per 64 keys and wave: 32 products, 370 vector
// instructions, a third of them the parts of P) and, per workgroup, by the
// chain of one tile.  Eight chunks of 200 to 512 tokens over prefixes of up
// to 3000, bf16 pages of 64, 32 heads over 8: 119 us with the append, 355 TFLOP/s
// of the causal products, against 2300 us row by row; four first prompts of 37 to
// 511 tokens, f32 pages of 64, 8 heads: 30.5 against 76 us.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "../host/status.hpp"
#include "../pool.hpp"
#include "bf16_parts.hpp"
#include "codecs.hpp"
#include "prefill_common.hpp"
#include "prefill_rank.hpp"
#include "prefill_tiles.hpp"

namespace airkv {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;
static_assert(kThreads == kRankThreads, "the ranking runs over the workgroup");

// Page types the kernel is built for: f32, bf16, and both 1-byte types (told
// apart at run time).
enum { kF32 = 0, kBf16 = 1, kByte = 2 };

// Shape of one instantiation.  D: head_dim rounded up to one of the built
// sizes (the columns past head_dim are staged as zeros).  NK: waves sharing a
// column set's keys.
template <int D, int PT, int NK> struct Shape {
    static constexpr int NP = PT == kBf16 ? 1 : 3;               // bf16 parts of a key or value
    static constexpr int COLS = 32 * kWaves / NK;                // (row, head) columns per workgroup
    static constexpr int SUB = NP == 1 && NK == 1 && D <= 128 ? 2 : 1;   // 32-key sub-tiles per wave and tile
    static constexpr int KT = 32 * SUB * NK;                     // keys per tile
    // K rows start 4 banks apart, V rows 16 banks apart (a transposing read
    // covers 4 rows x 64 bytes)
    static constexpr int KP = D * 2 + 16;
    static constexpr int VP = (D * 2) % 256 == 192 ? D * 2 : D * 2 + 64;
    static constexpr int KPART = KT * KP, VPART = KT * VP;       // one part of a K / V tile
    static constexpr int STAGE = NP * (KPART + VPART);
    static constexpr int BUFS = 2 * STAGE <= 144 * 1024 ? 2 : 1;
    static constexpr int LDS = BUFS * STAGE;
    static constexpr int CHUNKS = KT * (D / 8);                  // 8-element chunks of a K (or V) tile
    static constexpr int PASSES = (CHUNKS + kThreads - 1) / kThreads;
    static constexpr int MERGE = D * 128 + 512;                  // one wave's partial result
    static_assert((VP / 4) % 64 == 16 || (VP / 4) % 64 == 48, "V pitch: rows 16 banks apart");
    static_assert(LDS <= 160 * 1024 && LDS >= kRankLdsBytes, "LDS of a CU; the ranking borrows it");
    static_assert((kWaves - kWaves / NK) * MERGE <= LDS, "the waves' partial results fit");
};

__device__ __forceinline__ f32x16 mfma_bf16(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b),
                                                   c, 0, 0, 0);
}
// Eight cache elements in registers as loaded.
template <int PT> struct Raw;
template <> struct Raw<kF32> { f32x4 a, b; };
template <> struct Raw<kBf16> { u32x4 w; };
template <> struct Raw<kByte> { u32x2 w; float s; };

// The chunk at byte `at` of the pages and its scale at byte `sat` of the scales.
template <int PT>
__device__ __forceinline__ void load_raw(const void *pages, const float *scales, uint64_t at, uint64_t sat,
                                         Raw<PT> &r) {
    const char *p = (const char *)pages + at;
    if constexpr (PT == kF32) {
        r.a = *reinterpret_cast<const f32x4 *>(p);
        r.b = *reinterpret_cast<const f32x4 *>(p + 16);
    } else if constexpr (PT == kBf16) {
        r.w = *reinterpret_cast<const u32x4 *>(p);
    } else {
        r.w = *reinterpret_cast<const u32x2 *>(p);
        r.s = *reinterpret_cast<const float *>((const char *)scales + sat);
    }
}

// One 1-byte code as f32, unscaled.
__device__ __forceinline__ float code_f32(bool fp8, uint32_t byte) {
    return fp8 ? fp8_decode(byte) : (float)(int32_t)(int8_t)byte;
}

template <int PT>
__device__ __forceinline__ void to_f32(const Raw<PT> &r, bool fp8, float (&x)[8]) {
#pragma clang fp contract(off)
    if constexpr (PT == kF32) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            x[j] = r.a[j];
            x[4 + j] = r.b[j];
        }
    } else if constexpr (PT == kByte) {
        if (fp8) {
#pragma unroll
            for (int j = 0; j < 8; ++j) x[j] = fp8_decode((r.w[j >> 2] >> (8 * (j & 3))) & 0xFFu) * r.s;
        } else {
#pragma unroll
            for (int j = 0; j < 8; ++j)
                x[j] = (float)(int32_t)(int8_t)((r.w[j >> 2] >> (8 * (j & 3))) & 0xFFu) * r.s;
        }
    }
}

// Element e of page row `row` (row = (block * n_kv + head) * block_size + offset).
template <int PT>
__device__ __forceinline__ float page_elem(const PrefillArgs &a, const void *pages, const float *scales,
                                           int64_t row, int e) {
#pragma clang fp contract(off)
    const int64_t i = row * a.head_dim + e;
    if constexpr (PT == kF32) return ((const float *)pages)[i];
    else if constexpr (PT == kBf16) return bf16_to_f32(((const uint16_t *)pages)[i]);
    else return code_f32(a.fp8, ((const uint8_t *)pages)[i]) *
                scales[row * (a.head_dim / a.scale_group) + e / a.scale_group];
}

// One query row and head by one wave in plain f32: keys 0 .. n_keys - 1,
// 64 at a time (a key per lane for the scores, a head_dim element per lane for
// the values), out-of-pool entries as zero keys and values.
template <int PT>
__device__ void slow_column(const PrefillArgs &a, const int32_t *tbl, int kh, int bs_log2, int64_t qrow, int h,
                            int n_keys) {
    const int lane = threadIdx.x & 63, d = a.head_dim, bs = a.block_size;
    const int64_t qo = (qrow * a.n_q_heads + h) * d;
    auto q_elem = [&](int e) {
        return a.q_dtype == AIR_KV_F32 ? ((const float *)a.q)[qo + e] : bf16_to_f32(((const uint16_t *)a.q)[qo + e]);
    };
    auto page_row = [&](uint32_t t) -> int64_t {
        const int32_t blk = tbl[t >> bs_log2];
        if (blk < 0 || blk >= a.num_blocks) return -1;
        return ((int64_t)blk * a.n_kv_heads + kh) * bs + (int)(t & (uint32_t)(bs - 1));
    };
    float m = -INFINITY, l = 0.0f, acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (uint32_t t0 = 0; t0 < (uint32_t)n_keys; t0 += 64) {      // (up to 2^31 - 1 keys)
        float s = -INFINITY;
        if (t0 + lane < (uint32_t)n_keys) {
            const int64_t row = page_row(t0 + lane);
            s = 0.0f;
            for (int e = 0; e < d; ++e)
                s += q_elem(e) * (row < 0 ? 0.0f : page_elem<PT>(a, a.k_pages, a.k_scales, row, e));
            s *= a.scale_log2;
        }
        float mt = s;
        for (int o = 32; o >= 1; o >>= 1) mt = fmaxf(mt, __shfl_xor(mt, o));
        const float m_new = fmaxf(m, mt);
        const float alpha = m == -INFINITY ? 0.0f : exp2f(m - m_new);
        const float p = s == -INFINITY ? 0.0f : exp2f(s - m_new);
        float ps = p;
        for (int o = 32; o >= 1; o >>= 1) ps += __shfl_xor(ps, o);
        l = l * alpha + ps;
        m = m_new;
        for (int i = 0; i < 4; ++i) acc[i] *= alpha;
        const int n = (uint32_t)n_keys - t0 < 64 ? (int)((uint32_t)n_keys - t0) : 64;
        for (int j = 0; j < n; ++j) {
            const float pj = __shfl(p, j);
            const int64_t row = page_row(t0 + j);
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (lane + 64 * i < d)
                    acc[i] += pj * (row < 0 ? 0.0f : page_elem<PT>(a, a.v_pages, a.v_scales, row, lane + 64 * i));
        }
    }
    const float inv = 1.0f / l;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (lane + 64 * i >= d) break;
        if (a.out_dtype == AIR_KV_F32) ((float *)a.out)[qo + lane + 64 * i] = acc[i] * inv;
        else ((uint16_t *)a.out)[qo + lane + 64 * i] = bf16_rne(acc[i] * inv);
    }
}

// Waves per SIMD an instantiation is built for.
template <int D, int PT, int NK> constexpr int waves_per_simd() {
    return D >= 256 || Shape<D, PT, NK>::LDS > 80 * 1024 ? 1 : 2;
}

// NQ: bf16 parts of a query (1: bf16 queries, 3: f32).
template <int D, int PT, int NQ, int NK>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(waves_per_simd<D, PT, NK>())))
void prefill_f32_kernel(PrefillArgs a) {
    using S = Shape<D, PT, NK>;
    constexpr int KT = S::KT, SUB = S::SUB, KP = S::KP, VP = S::VP, PASSES = S::PASSES, NP = S::NP;
    __shared__ __align__(16) uint8_t smem[S::LDS];
    const int G = a.group, d = a.head_dim, nz = a.nz;
    const int row = (int)(blockIdx.x / (unsigned)a.n_kv_heads), kh = (int)(blockIdx.x % (unsigned)a.n_kv_heads);
    // Slot z of sequence b serves its work group n_wg - 1 - z and every nz-th
    // one below it; rows of the grid take the slots longest first.
    int b, z;
    // (a launch that is resident at once needs no order)
    if (a.batch == 1 || a.batch > kRankCap || (int64_t)a.batch * nz > kRankItems || (int)gridDim.x <= a.slots) {
        b = row % a.batch;
        z = row / a.batch;
    } else {
        const int item = rank_item(a, reinterpret_cast<int *>(smem), nz, row, [&](int64_t len, int64_t ql, int zz) {
            const int cols = (int)ql * G, n_wg = (cols + S::COLS - 1) / S::COLS;
            if (ql <= 0 || len < ql || zz >= n_wg) return (int64_t)0;
            const int end = (n_wg - zz) * S::COLS < cols ? (n_wg - zz) * S::COLS : cols;
            return len - ql + (end - 1) / G + 1;
        });
        b = item / nz;
        z = item - b * nz;
    }
    b = __builtin_amdgcn_readfirstlane(b);
    z = __builtin_amdgcn_readfirstlane(z);
    int32_t q0;
    int qlen;
    int64_t len;
    if (!prefill_begin<0, 0>(a, PrefillSlot{b, kh, z, 1, 0, 1, -1}, q0, qlen, len)) return;
    const int32_t *tbl = a.tables + (int64_t)b * a.max_blocks;
    const int bs_log2 = __builtin_ctz((unsigned)a.block_size), bs_mask = a.block_size - 1;
    const int sg_log2 = a.scale_group ? __builtin_ctz((unsigned)a.scale_group) : 0;
    const int n_sc = a.scale_group ? d >> sg_log2 : 0;
    const int q_offset = (int)(len - qlen);
    const int nc = qlen * G;                                    // columns of this (sequence, kv head)
    const int n_wg = (nc + S::COLS - 1) / S::COLS;
    const int tid = threadIdx.x, lane = tid & 63, r32 = lane & 31, hh = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int cg = wave / NK, kg = wave % NK;                   // column set, share of its keys

    // Staging: thread tid moves chunks tid + 256 i of a tile, chunk = 8
    // elements of one row.  Loads are unconditional (an id outside the pool
    // reads block 0, a column past head_dim column 0); what is not live is
    // staged as zeros.
    Raw<PT> rk[PASSES], rv[PASSES];
    int32_t id[PASSES];
    uint32_t live = 0;
    int rows = 0;                                               // NK > 1: rows past these are no wave's, left alone
    auto chunk_row = [&](int i) { return (tid + kThreads * i) / (D / 8); };
    auto chunk_col = [&](int i) { return (tid + kThreads * i) % (D / 8) * 8; };
    // A chunk keeps its place within its block (KT is a multiple of the block
    // size): byte offsets in a block, of elements and of scales.
    constexpr int EB = PT == kF32 ? 4 : PT == kBf16 ? 2 : 1;
    static_assert(KT % 32 == 0, "whole blocks of 16 or 32 tokens per tile");
    const uint32_t blk_bytes = (uint32_t)a.n_kv_heads * a.block_size * d * EB;
    const uint32_t blk_sc = (uint32_t)a.n_kv_heads * a.block_size * n_sc * 4;
    uint32_t off[PASSES], soff[PASSES];
#pragma unroll
    for (int i = 0; i < PASSES; ++i) {
        const uint32_t r = kh * a.block_size + (chunk_row(i) & bs_mask);
        const uint32_t col = chunk_col(i) < d ? chunk_col(i) : 0;
        off[i] = (r * d + col) * EB;
        soff[i] = PT == kByte ? (r * n_sc + (col >> sg_log2)) * 4 : 0;
    }
    auto fetch_ids = [&](int t, int kend) {
#pragma unroll
        for (int i = 0; i < PASSES; ++i) {
            const uint32_t j = entry_key(t, KT, chunk_row(i), kend) >> bs_log2;
            id[i] = *reinterpret_cast<const int32_t *>((const char *)tbl + 4 * j);
        }
    };
    auto load_tile = [&](int t, int kend) {
        live = 0;
        rows = tile_rows(t, KT, kend);
#pragma unroll
        for (int i = 0; i < PASSES; ++i) {
            if (NK > 1 && chunk_row(i) >= rows) continue;
            const bool in_pool = id[i] >= 0 && id[i] < a.num_blocks;
            if (tile_key(t, KT, chunk_row(i)) < (uint32_t)kend && in_pool && chunk_col(i) < d) live |= 1u << i;
            const uint32_t blk = in_pool ? id[i] : 0;
            const uint64_t at = (uint64_t)blk * blk_bytes + off[i], sat = (uint64_t)blk * blk_sc + soff[i];
            load_raw<PT>(a.k_pages, a.k_scales, at, sat, rk[i]);
            load_raw<PT>(a.v_pages, a.v_scales, at, sat, rv[i]);
        }
    };
    auto stage_tile = [&](int buf) {
        uint8_t *ks = smem + buf * S::STAGE, *vs = ks + NP * S::KPART;
#pragma unroll
        for (int i = 0; i < PASSES; ++i) {
            if (S::CHUNKS % kThreads != 0 && tid + kThreads * i >= S::CHUNKS) break;
            if (NK > 1 && chunk_row(i) >= rows) continue;
            const bool lv = (live >> i) & 1;
            uint8_t *kd = ks + chunk_row(i) * KP + chunk_col(i) * 2;
            uint8_t *vd = vs + chunk_row(i) * VP + chunk_col(i) * 2;
            const u32x4 zero = {0, 0, 0, 0};
            if constexpr (NP == 1) {
                *reinterpret_cast<u32x4 *>(kd) = lv ? rk[i].w : zero;
                *reinterpret_cast<u32x4 *>(vd) = lv ? rv[i].w : zero;
            } else {
                auto put = [&](const Raw<PT> &r, uint8_t *dst, int part) {
                    float x[8];
                    to_f32<PT>(r, a.fp8, x);
                    u32x4 p[3];
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        uint32_t h, m, l;
                        split3(x[2 * j], x[2 * j + 1], h, m, l);
                        p[0][j] = h;
                        p[1][j] = m;
                        p[2][j] = l;
                    }
#pragma unroll
                    for (int c = 0; c < 3; ++c) *reinterpret_cast<u32x4 *>(dst + c * part) = lv ? p[c] : zero;
                };
                put(rk[i], kd, S::KPART);
                put(rv[i], vd, S::VPART);
            }
        }
    };

    for (int w = z; w < n_wg; w += nz) {
        const int c0 = (n_wg - 1 - w) * S::COLS;                // the workgroup's first column
        const int c_end = c0 + S::COLS < nc ? c0 + S::COLS : nc;
        const int kend = q_offset + (c_end - 1) / G + 1;        // keys the workgroup needs
        const int nt = key_tiles(kend, KT);
        const int wc = c0 + 32 * cg;                        // the wave's first column
        const bool wlive = wc < c_end;
        const int col = wc + r32 < c_end ? wc + r32 : c_end - 1;
        const int qr = col / G, h = kh * G + col - qr * G;
        const int qpos = q_offset + qr;
        // the wave's positions: tiles at or past the end are skipped, tiles
        // below the first need no mask (uniform)
        const uint32_t pos_end = __builtin_amdgcn_readfirstlane(
            wlive ? q_offset + (wc + 31 < c_end ? wc + 31 : c_end - 1) / G + 1 : 0);
        const uint32_t pos_lo = __builtin_amdgcn_readfirstlane(q_offset + (wlive ? wc : c_end - 1) / G);

        fetch_ids(0, kend);
        // ---- queries, in the B operand's layout (column r32)
        u32x4 qp[NQ][D / 16];                                   // parts: head_dim 16 ks + 8 hh .. + 8
        {
            const int64_t qo = ((int64_t)(q0 + qr) * a.n_q_heads + h) * d;
            if constexpr (NQ == 1) {
#pragma unroll
                for (int ks = 0; ks < D / 16; ++ks) {
                    qp[0][ks] = u32x4{0, 0, 0, 0};
                    if (16 * ks < d)
                        qp[0][ks] = *reinterpret_cast<const u32x4 *>((const uint16_t *)a.q + qo + 16 * ks + 8 * hh);
                }
            } else {
#pragma unroll
                for (int ks = 0; ks < D / 16; ++ks) {
                    f32x4 x = {0.0f, 0.0f, 0.0f, 0.0f}, y = x;
                    if (16 * ks < d) {
                        const f32x4 *src = reinterpret_cast<const f32x4 *>((const float *)a.q + qo + 16 * ks + 8 * hh);
                        x = src[0];
                        y = src[1];
                    }
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const f32x4 v = j < 2 ? x : y;
                        uint32_t hi, mid, lo;
                        split3(v[2 * (j & 1)], v[2 * (j & 1) + 1], hi, mid, lo);
                        qp[0][ks][j] = hi;
                        qp[1][ks][j] = mid;
                        qp[2][ks][j] = lo;
                    }
                }
            }
        }

        f32x16 acc[D / 32];                                     // O^T: column r32, head_dim 32 n + 8 (i / 4) + 4 hh + i % 4
#pragma unroll
        for (int n = 0; n < D / 32; ++n)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[n][i] = 0.0f;
        float m_run = -INFINITY, l_run = 0.0f;

        // S^T of the 32 keys from row kb of the staged tile: lane holds keys
        // 8 (i / 4) + 4 hh + i % 4 of its column
        auto scores = [&](const uint8_t *ks, int kb) {
            // chains: the leading part products (two of them past 64
            // elements), and the others' sum
            f32x16 s0, s1, sl;
#pragma unroll
            for (int i = 0; i < 16; ++i) s0[i] = s1[i] = sl[i] = 0.0f;
            const uint8_t *kr = ks + (kb + r32) * KP + 16 * hh;
#pragma unroll
            for (int k = 0; k < D / 16; ++k) {
                u32x4 kA[NP];
#pragma unroll
                for (int c = 0; c < NP; ++c) kA[c] = *reinterpret_cast<const u32x4 *>(kr + c * S::KPART + 32 * k);
#pragma unroll
                for (int o = 2; o >= 1; --o)                     // part products of order 2^-8o
#pragma unroll
                    for (int c = 0; c < NP; ++c)
                        if (o - c >= 0 && o - c < NQ) sl = mfma_bf16(kA[c], qp[o - c][k], sl);
                if (D > 64 && (k & 1)) s1 = mfma_bf16(kA[0], qp[0][k], s1);
                else s0 = mfma_bf16(kA[0], qp[0][k], s0);
            }
            if constexpr (D > 64) s0 += s1;
            if constexpr (NP > 1 || NQ > 1) s0 += sl;
            return s0;
        };
        // o (+)= V^T . P^T over the 32 keys from row kb (`first`: from zero)
        f32x16 o[D / 32];
        auto add_values = [&](const uint8_t *vs, int kb, const float (&p)[16], bool first) {
            u32x4 pp[3][2];                                      // parts of P: keys 16 st + 4 hh + (0..3, 8..11)
#pragma unroll
            for (int st = 0; st < 2; ++st)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    uint32_t h, m, l;
                    split3(p[8 * st + 2 * j], p[8 * st + 2 * j + 1], h, m, l);
                    pp[0][st][j] = h;
                    pp[1][st][j] = m;
                    pp[2][st][j] = l;
                }
            // two transposing reads per 16 keys: lane 16 g + s points at V[key
            // 4 hh + s / 4][16 (g % 2) + 4 (s % 4)] and receives four
            // consecutive keys of one head_dim column
            const int sl = lane & 15;
            const uint8_t *vr = vs + (kb + 4 * hh + (sl >> 2)) * VP + 2 * (16 * ((lane >> 4) & 1) + 4 * (sl & 3));
#pragma unroll
            for (int n = 0; n < D / 32; ++n) {
                if (first)
#pragma unroll
                    for (int i = 0; i < 16; ++i) o[n][i] = 0.0f;
                u32x4 va[NP][2];
#pragma unroll
                for (int c = 0; c < NP; ++c)
#pragma unroll
                    for (int st = 0; st < 2; ++st) {
                        const uint8_t *at = vr + c * S::VPART + 16 * st * VP + 64 * n;
                        const s16x4 t0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                            (__attribute__((address_space(3))) s16x4 *)(at));
                        const s16x4 t1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                            (__attribute__((address_space(3))) s16x4 *)(at + 8 * VP));
                        const u32x2 a0 = __builtin_bit_cast(u32x2, t0), a1 = __builtin_bit_cast(u32x2, t1);
                        va[c][st] = u32x4{a0[0], a0[1], a1[0], a1[1]};
                    }
#pragma unroll
                for (int od = 2; od >= 0; --od)                  // part products of order 2^-8od, the least first
#pragma unroll
                    for (int c = 0; c < NP; ++c)
                        if (od - c >= 0)
#pragma unroll
                            for (int st = 0; st < 2; ++st) o[n] = mfma_bf16(va[c][st], pp[od - c][st], o[n]);
            }
        };
        auto compute_tile = [&](int t) {
            const uint8_t *ks = smem + (S::BUFS == 2 ? (t & 1) * S::STAGE : 0), *vs = ks + NP * S::KPART;
            const int kb = 32 * SUB * kg;                        // the wave's first key: of the tile, of the sequence
            const uint32_t k0 = tile_key(t, KT, kb);
            if (k0 >= pos_end) return;                           // behind every row of the wave (uniform)
            f32x16 s[SUB];
#pragma unroll
            for (int u = 0; u < SUB; ++u) s[u] = scores(ks, kb + 32 * u);
            if (k0 + 32 * SUB - 1 > pos_lo) {
#pragma unroll
                for (int u = 0; u < SUB; ++u) {
                    const int kq = (int)((uint32_t)qpos - k0) - 32 * u - 4 * hh;
#pragma unroll
                    for (int i = 0; i < 16; ++i) s[u][i] = 8 * (i >> 2) + (i & 3) <= kq ? s[u][i] : -INFINITY;
                }
            }
            float mt = s[0][0];
#pragma unroll
            for (int u = 0; u < SUB; ++u)
#pragma unroll
                for (int i = 0; i < 16; ++i) mt = fmaxf(mt, s[u][i]);
            const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(mt), __float_as_uint(mt), false, false);
            mt = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1])) * a.scale_log2;
            // the running max follows only when a tile exceeds it by 2^8: the
            // probabilities stay below 256 and most tiles skip the rescale
            if (__ballot(mt > m_run + 8.0f) != 0ull) {
                const float m_new = fmaxf(m_run, mt);
                const float alpha = m_run == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_run - m_new);
                l_run *= alpha;
#pragma unroll
                for (int n = 0; n < D / 32; ++n) acc[n] *= alpha;
                m_run = m_new;
            }
            const float mu = m_run == -INFINITY ? 0.0f : m_run;   // no key seen yet: every p is 0
#pragma unroll
            for (int u = 0; u < SUB; ++u) {
                float p[16];
#pragma unroll
                for (int i = 0; i < 16; ++i) p[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[u][i], a.scale_log2, -mu));
                float l4[4] = {p[0], p[1], p[2], p[3]};
#pragma unroll
                for (int i = 4; i < 16; ++i) l4[i & 3] += p[i];
                l_run += (l4[0] + l4[1]) + (l4[2] + l4[3]);
                add_values(vs, kb + 32 * u, p, u == 0);
            }
#pragma unroll
            for (int n = 0; n < D / 32; ++n) acc[n] += o[n];
        };

        load_tile(0, kend);
        fetch_ids(1, kend);
        if constexpr (S::BUFS == 2) {
            stage_tile(0);
            if (nt > 1) {
                load_tile(1, kend);
                fetch_ids(2, kend);
            }
            __syncthreads();
            for (int t = 0; t < nt; ++t) {
                compute_tile(t);
                if (t + 1 < nt) stage_tile((t + 1) & 1);
                __syncthreads();
                if (t + 2 < nt) {
                    load_tile(t + 2, kend);
                    fetch_ids(t + 3, kend);
                }
            }
        } else {
            for (int t = 0; t < nt; ++t) {
                stage_tile(0);
                __syncthreads();
                if (t + 1 < nt) {
                    load_tile(t + 1, kend);
                    fetch_ids(t + 2, kend);
                }
                compute_tile(t);
                __syncthreads();
            }
        }

        // ---- the key shares of a column set, folded into its first wave
        float l = l_run + __shfl_xor(l_run, 32);
        if constexpr (NK > 1) {
            // the shares past the first go to LDS (the last tile's barrier has
            // freed it), the first folds them
            if (kg > 0) {
                uint8_t *at = smem + (cg * (NK - 1) + kg - 1) * S::MERGE;
                f32x4 *po = reinterpret_cast<f32x4 *>(at) + lane;
#pragma unroll
                for (int n = 0; n < D / 32; ++n)
#pragma unroll
                    for (int i4 = 0; i4 < 4; ++i4)
                        po[(4 * n + i4) * 64] = f32x4{acc[n][4 * i4], acc[n][4 * i4 + 1], acc[n][4 * i4 + 2],
                                                      acc[n][4 * i4 + 3]};
                // both lanes of a column hold the same max and sum
                reinterpret_cast<float *>(at + D * 128)[lane] = hh ? l : m_run;
            }
            __syncthreads();
            if (kg == 0) {
#pragma unroll
                for (int g = 0; g < NK - 1; ++g) {
                    const uint8_t *at = smem + (cg * (NK - 1) + g) * S::MERGE;
                    const f32x4 *po = reinterpret_cast<const f32x4 *>(at) + lane;
                    const float *ml = reinterpret_cast<const float *>(at + D * 128) + r32;
                    const float om = ml[0], ol = ml[32];
                    const float m_new = fmaxf(m_run, om);
                    const float sa = m_run == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_run - m_new);
                    const float sb = om == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(om - m_new);
                    l = l * sa + ol * sb;
#pragma unroll
                    for (int n = 0; n < D / 32; ++n)
#pragma unroll
                        for (int i4 = 0; i4 < 4; ++i4) {
                            const f32x4 o = po[(4 * n + i4) * 64];
#pragma unroll
                            for (int e = 0; e < 4; ++e) acc[n][4 * i4 + e] = acc[n][4 * i4 + e] * sa + o[e] * sb;
                        }
                    m_run = m_new;
                }
            }
        }
        if (kg == 0 && wlive) {
            const bool mine = wc + r32 < c_end;
            const float inv = 1.0f / l;
            float sum = 0.0f;                                    // finite unless some output is not
#pragma unroll
            for (int n = 0; n < D / 32; ++n)
#pragma unroll
                for (int i = 0; i < 16; ++i) sum += acc[n][i] * inv;
            if (mine) {
                const int64_t oo = ((int64_t)(q0 + qr) * a.n_q_heads + h) * d + 4 * hh;
#pragma unroll
                for (int n = 0; n < D / 32; ++n) {
                    if (32 * n >= d) break;
#pragma unroll
                    for (int i4 = 0; i4 < 4; ++i4) {
                        const f32x4 v = f32x4{acc[n][4 * i4], acc[n][4 * i4 + 1], acc[n][4 * i4 + 2],
                                              acc[n][4 * i4 + 3]} * inv;
                        if (a.out_dtype == AIR_KV_F32) {
                            *reinterpret_cast<f32x4 *>((float *)a.out + oo + 32 * n + 8 * i4) = v;
                        } else {
                            *reinterpret_cast<u32x2 *>((uint16_t *)a.out + oo + 32 * n + 8 * i4) =
                                u32x2{(uint32_t)bf16_rne(v[0]) | ((uint32_t)bf16_rne(v[1]) << 16),
                                      (uint32_t)bf16_rne(v[2]) | ((uint32_t)bf16_rne(v[3]) << 16)};
                        }
                    }
                }
            }
            const uint64_t bad = __ballot(mine && !__builtin_isfinite(sum));
            uint32_t redo = (uint32_t)bad | (uint32_t)(bad >> 32);
            if (redo) __builtin_amdgcn_s_waitcnt(0);             // the stores above land before their replacements
            while (redo) {
                const int c = __builtin_ctz(redo);
                redo &= redo - 1;
                const int rr = (wc + c) / G;
                slow_column<PT>(a, tbl, kh, bs_log2, (int64_t)q0 + rr, kh * G + wc + c - rr * G, q_offset + rr + 1);
            }
        }
        __syncthreads();                                         // the next work group restages LDS
    }
    // the out-of-pool table entries within the sequence's length, once per sequence
    if (z == 0 && kh == 0) {
        for (int64_t j = threadIdx.x; j < (len + a.block_size - 1) >> bs_log2; j += kThreads) {
            const int32_t blk = tbl[j];
            if (blk < 0 || blk >= a.num_blocks) atomicAdd(a.errors, 1ull);
        }
    }
}

template <int D, int PT, int NQ, int NK>
hipError_t launch_one(PrefillArgs a, int64_t nz, hipStream_t s) {
    // a dispatch counts its work-items in 32 bits: at most 2^32 / 256 - 1
    // workgroups (fewer slots per sequence only lengthen each slot's stride)
    const int64_t cap = ((int64_t)0xffffffff / kThreads) / ((int64_t)a.batch * a.n_kv_heads);
    nz = nz > cap ? cap : nz;
    if (nz < 1) return hipErrorInvalidConfiguration;
    a.nz = (int32_t)nz;
    hipLaunchKernelGGL((prefill_f32_kernel<D, PT, NQ, NK>), dim3((unsigned)((int64_t)a.batch * a.n_kv_heads * nz)),
                       dim3(kThreads), 0, s, a);
    return hipGetLastError();
}

// Key shares per column set: 4 or 2 where the launch would otherwise leave
// waves or compute units idle -- a chunk whose columns fill no more than 128 /
// NK (the other waves of the workgroup would have none), or a launch that
// is still resident at once with its workgroups NK times as many -- and where a tile of NK times 32 keys fits LDS.
template <int D, int PT, int NQ>
hipError_t launch_nk(const PrefillArgs &a, int32_t max_q_len, hipStream_t s) {
    constexpr int kMost = D <= 96 ? 4 : D <= 128 || PT == kBf16 ? 2 : 1;
    const int64_t cols = (int64_t)(max_q_len > 0 ? max_q_len : 1) * a.group;
    const int64_t per_seq = (int64_t)a.batch * a.n_kv_heads;
    auto slots = [&](int nk) { return (cols * nk + 32 * kWaves - 1) / (32 * kWaves); };
    // resident: workgroups of an instantiation the GPU holds at once
    auto use = [&](int nk, int resident) { return slots(nk) == 1 || per_seq * slots(nk) <= resident; };
    if constexpr (kMost >= 4)
        if (use(4, a.slots * waves_per_simd<D, PT, 4>())) return launch_one<D, PT, NQ, 4>(a, slots(4), s);
    if constexpr (kMost >= 2)
        if (use(2, a.slots * waves_per_simd<D, PT, 2>())) return launch_one<D, PT, NQ, 2>(a, slots(2), s);
    return launch_one<D, PT, NQ, 1>(a, slots(1), s);
}

template <int D>
hipError_t launch_d(const PrefillArgs &a, int dtype, int32_t max_q_len, hipStream_t s) {
    const bool qf32 = a.q_dtype == AIR_KV_F32;
    if (dtype == AIR_KV_F32)
        return qf32 ? launch_nk<D, kF32, 3>(a, max_q_len, s) : launch_nk<D, kF32, 1>(a, max_q_len, s);
    // the matrix-core kernel of paged_prefill.hip has the other pages of 128
    if constexpr (D == 128) return hipErrorInvalidValue;
    else if (dtype == AIR_KV_BF16)
        return qf32 ? launch_nk<D, kBf16, 3>(a, max_q_len, s) : launch_nk<D, kBf16, 1>(a, max_q_len, s);
    else return qf32 ? launch_nk<D, kByte, 3>(a, max_q_len, s) : launch_nk<D, kByte, 1>(a, max_q_len, s);
}

}  // namespace

hipError_t launch_prefill_f32(PrefillArgs a, int dtype, int32_t max_q_len, int cus, hipStream_t s) {
    a.max_len = (int64_t)a.max_blocks * a.block_size;
    a.ns_max = 1;
    a.slots = cus;                                              // compute units
    a.fp8 = dtype == AIR_KV_FP8;
    if (a.head_dim <= 64) return launch_d<64>(a, dtype, max_q_len, s);
    if (a.head_dim <= 96) return launch_d<96>(a, dtype, max_q_len, s);
    if (a.head_dim == 128) return launch_d<128>(a, dtype, max_q_len, s);
    return launch_d<256>(a, dtype, max_q_len, s);
}

}  // namespace airkv
