// Paged decode: validation of a launch's shape and the choice of its kernel
// (paged_decode_mfma.hip, or paged_decode_f32.hip for the pools and groups
// that one does not take).
#include <hip/hip_runtime.h>

#include "../host/status.hpp"
#include "../pool.hpp"
#include "decode_common.hpp"

namespace airkv {

int plan_decode(const air_kv_pool &p, int32_t n_q_heads, int32_t batch, int32_t max_blocks,
                int32_t max_splits, DecodePlan *plan) {
    const int nkv = p.desc.n_kv_heads, d = p.desc.head_dim, bs = p.desc.block_size;
    if (n_q_heads <= 0 || n_q_heads % nkv)
        return fail(AIR_KV_E_INVALID_ARG, "n_q_heads %d is not a multiple of n_kv_heads %d", n_q_heads, nkv);
    const int g = n_q_heads / nkv;
    if (!decode_mfma_supported(p.desc.dtype, d, bs, g, p.desc.scale_group)) {
        if (d <= 0 || d % 8 || d > 256)
            return fail(AIR_KV_E_INVALID_ARG, "decode supports head_dim a multiple of 8 up to 256 (pool has %d)", d);
    }
    if (batch < 0 || batch > 65535) return fail(AIR_KV_E_INVALID_ARG, "batch %d out of range", batch);
    if (max_blocks <= 0) return fail(AIR_KV_E_INVALID_ARG, "max_blocks must be positive");
    if (max_splits < 1 || max_splits > 256)
        return fail(AIR_KV_E_INVALID_ARG, "max_splits %d outside 1..256", max_splits);
    plan->group = g;
    plan->max_splits = max_splits;
    if (decode_mfma_supported(p.desc.dtype, d, bs, g, p.desc.scale_group))
        return plan_decode_mfma(p, n_q_heads, batch, max_blocks, max_splits, plan);
    return plan_decode_f32(p, n_q_heads, batch, max_blocks, max_splits, plan);
}

hipError_t launch_decode(const air_kv_pool &p, hipStream_t s, const DecodePlan &plan, const void *q,
                         int32_t q_dtype, int32_t n_q_heads, const int32_t *tables,
                         const int32_t *lens, int32_t batch, int32_t max_blocks, float scale,
                         void *workspace, void *out, int32_t out_dtype, const float *k_new,
                         const float *v_new) {
    DecodeArgs a;
    a.k_new = k_new;
    a.v_new = v_new;
    a.q = q; a.q_dtype = q_dtype; a.n_q_heads = n_q_heads;
    a.tables = tables; a.lens = lens;
    a.batch = batch; a.max_blocks = max_blocks;
    const int waves = p.desc.n_kv_heads * ((plan.group + 15) / 16);   // per slice
    a.simd_slices = (4 * p.cus + waves - 1) / waves;
    a.slices = plan.slices; a.slots = plan.slots; a.max_splits = plan.max_splits;
    a.seq_pieces = plan.seq_pieces;
    a.scale_log2 = scale * 1.4426950408889634f;
    a.n_kv_heads = p.desc.n_kv_heads; a.block_size = p.desc.block_size;
    a.scale_group = p.desc.scale_group; a.group = plan.group; a.num_blocks = p.desc.num_blocks;
    a.k_pages = p.k_pages; a.v_pages = p.v_pages;
    a.k_scales = p.k_scales; a.v_scales = p.v_scales;
    a.out = out; a.out_dtype = out_dtype;
    a.errors = p.errors;
    a.prefix = nullptr;
    a.part_o = a.part_ml = nullptr;
    a.head_dim = p.desc.head_dim;
    return plan.mfma ? launch_decode_mfma(a, plan, workspace, s) : launch_decode_f32(a, plan, workspace, s);
}

}  // namespace airkv
