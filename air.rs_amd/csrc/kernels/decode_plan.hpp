// Arithmetic of the decode kernels' work division, in host and device code, so
// that it can be checked on the CPU (tests/decode_plan_check.cpp).
#pragma once

#include <math.h>
#include <stddef.h>
#include <stdint.h>

#ifdef __HIPCC__
#define AIRKV_HD __host__ __device__
#else
#define AIRKV_HD
#endif

namespace airkv {

constexpr int kMaxBatch = 4096;            // sequences per launch (the host splits larger batches)

// ceil(n / m) of counts up to 2^31 - 1.
AIRKV_HD inline int ceil_div(int n, int m) { return (int)(((uint32_t)n + (uint32_t)m - 1) / (uint32_t)m); }

// Tiles per slice: an equal share of `total` over the resident waves, but at
// least full_chunk once every SIMD has a wave (simd_slices per kv head), and
// large enough that no sequence meets more than max_splits slices.  A sequence
// of T tiles starting anywhere meets at most ceil((T - 1) / chunk) + 1 slices, so
// chunk >= ceil((T - 1) / (max_splits - 1)) for the longest sequence (tmax tiles)
// bounds every one; max_splits 1 leaves one slice per kv head.
AIRKV_HD inline int slice_chunk(int total, int slices, int simd_slices, int full_chunk, int tmax, int max_splits) {
    const int lone = ceil_div(total, simd_slices);
    int c = ceil_div(total, slices);
    const int least = lone < full_chunk ? lone : full_chunk;
    c = c > least ? c : least;
    c = c > 1 ? c : 1;
    if (max_splits <= 1) return c > total ? c : total;
    const int cs = (tmax - 1 + max_splits - 2) / (max_splits - 1);
    return c > cs ? c : cs;
}

// The f32-precision decode counts max_splits in partitions, and up to kSharing
// slices share one as long as they keep shared_tiles(t) tiles, t the tiles of
// the sequence: a tile is about 1.6 us of a slice, a partial row 0.1 (head_dim 64)
// to 0.25 us (256) of the merge, so c tiles a slice and t / c rows cost least near
// c = sqrt(t / 6).  (The vector kernel before it gave a partition four waves.)
constexpr int kSharing = 4;
AIRKV_HD inline int shared_tiles(int t) {
    const int c = (int)sqrtf((float)t * (1.0f / 6));
    return c > 2 ? c : 2;
}

// Its tiles per slice (max_splits at least 2; simd_slices give every SIMD a wave).
AIRKV_HD inline int shared_chunk(int total, int slices, int simd_slices, int tmax, int max_splits) {
    int c = ceil_div(total, slices);
    c = c > 1 ? c : 1;
    const int part = (tmax - 1 + max_splits - 2) / (max_splits - 1);          // slice_chunk's, by partitions
    if (part <= c) return c;
    const int most = max_splits * kSharing - 1;
    int cs = (tmax - 1 + most - 1) / most;                                    // and by their slices
    cs = cs > shared_tiles(tmax) ? cs : shared_tiles(tmax);
    // a few slices more than SIMDs: the SIMDs with two would end last
    const int lone = ceil_div(total, simd_slices);
    if (cs < lone && cs > lone / 3 * 2) cs = lone;
    cs = cs < part ? cs : part;
    return c > cs ? c : cs;
}

// Tiles per slice of a sequence of `tiles` tiles that has `pieces` slices of its own.
AIRKV_HD inline int piece_tiles(int tiles, int pieces) {
    const int c = (tiles + pieces - 1) / pieces;
    return c > shared_tiles(tiles) ? c : shared_tiles(tiles);
}

// The row of a cut sequence's partial result (f32-precision decode): sequence
// b's piece in slice w, `starts` if it is the sequence's first.  The cut pieces
// of a launch in order have increasing rows (a slice holds at most two, the end
// of one sequence and the start of another), all below slices + min(batch,
// slices): what the launch can cut, not what the batch holds.
AIRKV_HD inline int part_row(int w, int b, bool starts) {
    const int at = w + (starts ? 1 : 0);
    return w + (b < at ? b : at);
}
AIRKV_HD inline int64_t part_rows(int64_t slices, int64_t batch) { return slices + (batch < slices ? batch : slices); }

constexpr size_t kWsBytes = (size_t)32 << 20;

// Launch shape of the f32-precision decode.
struct DecodeF32Plan {
    int64_t batch;                     // sequences per launch
    int64_t slices, slices_qf32;       // slices per kv head under bf16 and under f32 queries
    int64_t seq_pieces;                // 0: slices of the batch's tiles; else each sequence has this many of its own
    int64_t slots;                     // partial rows per query head
    size_t ws_bytes;
};

inline size_t decode_align256(size_t x) { return (x + 255) & ~(size_t)255; }

// One slice for every wave slot of the GPU (waves / waves_qf32 slices' worth
// under bf16 / f32 queries, per_slice of them to a slice of all heads), and no
// more than keep the workspace within 32 MB (air_paged_decode_noalloc's array)
// or what one partial result per query head, sequence and 256 tokens takes (many
// query heads over few kv heads would otherwise ask for hundreds of megabytes).
//
// max_splits 1 gives each sequence slices of its own, so that its result does not
// depend on the others.
inline DecodeF32Plan plan_f32(int64_t n_q_heads, int64_t per_slice, int64_t d, int64_t block_size, int64_t batch,
                              int64_t max_blocks, int64_t max_splits, int64_t waves, int64_t waves_qf32) {
    auto min64 = [](int64_t a, int64_t b) { return a < b ? a : b; };
    auto max64 = [](int64_t a, int64_t b) { return a > b ? a : b; };
    // lengths are 32-bit: a wider table's rest is never reached
    const int64_t tiles_per_seq = max64(1, min64((max_blocks * block_size + 15) / 16, ((int64_t)INT32_MAX + 15) / 16));
    DecodeF32Plan pl;
    // tiles of a launch in 32 bits, with room for the windows of 64 past the last
    const int64_t nb = pl.batch = max64(1, min64(min64(batch, kMaxBatch), (INT32_MAX - 65536) / tiles_per_seq));
    const int64_t parts = min64(max_splits, (tiles_per_seq + 15) / 16);
    const size_t row = (size_t)n_q_heads * (d + 2) * 4, wide = row * nb * parts;
    const size_t rest = decode_align256((size_t)(nb + 2) * 4) + 256;     // the prefix and the alignment of the sums
    const int64_t rows = (int64_t)(((wide > kWsBytes ? wide : kWsBytes) - rest) / row);
    const int64_t fit = max64(1, max64(rows - nb, rows / 2));           // the most slices whose part_rows are at most `rows`
    const int64_t cuts = nb * min64(max_splits * kSharing, tiles_per_seq);
    auto slices_for = [&](int64_t w) { return min64(min64((w + per_slice - 1) / per_slice, cuts), fit); };
    if (max_splits > 1) {
        pl.seq_pieces = 0;
        // the bf16-query build runs at least as many waves: the workspace is its
        pl.slices = slices_for(waves);
        pl.slices_qf32 = min64(pl.slices, slices_for(waves_qf32));
        pl.slots = part_rows(pl.slices, nb);
    } else {
        pl.seq_pieces = max64(1, min64(min64(kSharing, rows / nb), (tiles_per_seq + 1) / 2));
        pl.slices = pl.slices_qf32 = pl.slots = nb * pl.seq_pieces;
        if (pl.seq_pieces == 1) pl.slots = 1;                           // no sequence is cut
    }
    pl.ws_bytes = decode_align256((size_t)(nb + 2) * 4) + decode_align256((size_t)n_q_heads * pl.slots * 2 * 4) +
                  (size_t)n_q_heads * pl.slots * d * 4;
    return pl;
}

}  // namespace airkv
