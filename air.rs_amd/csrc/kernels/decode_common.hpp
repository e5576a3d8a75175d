// Shared launch parameters of the paged decode kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

struct air_kv_pool;

namespace airkv {

struct DecodePlan;

// Everything a decode kernel needs; built once per launch on the host.
struct DecodeArgs {
    const void *q;
    int32_t q_dtype, n_q_heads;
    const int32_t *tables, *lens;
    int32_t batch, max_blocks;
    int32_t slices, slots;         // balanced slices per kv head, partial rows per (kv head, query head)
    int32_t simd_slices;           // slices per kv head that give every SIMD one wave
    int32_t max_splits;            // partitions of a sequence at most
    int32_t seq_pieces;            // f32-precision kernel: slices of each sequence's own (0: of the batch's tiles)
    float scale_log2;              // softmax scale * log2(e): exp(x*s) == exp2(x*scale_log2)
    int32_t n_kv_heads, block_size, scale_group, group, head_dim;
    int64_t num_blocks;
    const void *k_pages, *v_pages;
    const float *k_scales, *v_scales;
    // [n_kv][slots][group][head_dim] and [..][2]
    float *part_o;                 // unnormalised partial outputs
    float *part_ml;                // running max (log2 units), sum
    int32_t *prefix;               // tiles before each sequence, [batch + 1], then the chunk
    void *out;
    int32_t out_dtype;
    unsigned long long *errors;
    // The decode step's new K / V rows, [batch][n_kv_heads][head_dim] f32,
    // written as each sequence's token seq_lens[b] - 1 by the wave that
    // computes that token's tile (NULL: none)
    const float *k_new, *v_new;
};

bool decode_mfma_supported(int dtype, int head_dim, int block_size, int group, int scale_group);
int plan_decode_mfma(const air_kv_pool &p, int32_t n_q_heads, int32_t batch, int32_t max_blocks,
                     int32_t max_splits, DecodePlan *plan);
hipError_t launch_decode_mfma(const DecodeArgs &a, const DecodePlan &plan, void *workspace,
                              hipStream_t s);

int plan_decode_f32(const air_kv_pool &p, int32_t n_q_heads, int32_t batch, int32_t max_blocks,
                    int32_t max_splits, DecodePlan *plan);
hipError_t launch_decode_f32(const DecodeArgs &a, const DecodePlan &plan, void *workspace,
                             hipStream_t s);

}  // namespace airkv
