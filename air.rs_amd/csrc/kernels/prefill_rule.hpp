// Which kernel a prefill of the pools paged_prefill.hip does not take is faster
// on, from what the host knows of the launch.
#pragma once

#include <math.h>
#include <stdint.h>

#include "air_kv.h"

namespace airkv {

struct PrefillShape {
    int32_t dtype, head_dim, n_kv_heads, group, q_dtype;
    int32_t total_q, batch, max_q_len;
    int64_t tokens;                    // the table's width
};

// Whether paged_prefill_f32.hip beats paged_prefill_rows.hip (a workgroup per query
// row, kv head and eight heads of the group).  Both times are modelled as the
// longest row's chain of 64-key steps and the launch's work, joined as the sides
// of a right angle, and fitted to 1500 shapes measured on both kernels
// (profiles/prefill_f32_rule.csv: head_dim 32 to 256, every page type, 1 to 700
// rows, groups 1 to 8, prefixes 0 to 4000, 2 to 512 (sequence, kv head) pairs).  Taken
// together the choices lose 0.4% to the faster kernel; 11 of the 1500 are more than
// 3% slower than the rows.  Rows start sooner (one row without a prefix, head_dim
// 64: 4.1 us against 6.5; 256: 6 against 14) and f32 or 1-byte tiles are dear to
// split, but their work grows with the rows: eight 512-token chunks over bf16
// pages of 64 take 2300 us there against 127.  Sequence lengths are not known here,
// so the table's width stands for them; where it is wider than the chunk the
// prefix may be shorter, which favours the rows (factor 1.1 in place of 1.05).
inline bool prefill_f32_better(const PrefillShape &a) {
    const int64_t rows = a.max_q_len > 0 ? a.max_q_len : 1;
    if ((int64_t)a.total_q * a.group > INT32_MAX - 1024) return false;   // columns are counted in 32 bits
    const int64_t most = rows * a.batch, held = a.total_q < most ? a.total_q : most;
    const int64_t wgs = held * a.n_kv_heads * ((a.group + 7) / 8);
    if (wgs > 2560) return true;
    // steps of the longest row, of an average one
    const double steps = (double)((a.tokens + 63) / 64);
    double mean = ((double)a.tokens - (double)(rows - 1) / 2) / 64;
    mean = mean > 1.0 ? mean : 1.0;
    // us: {start, step} of a row's chain and of a workgroup's share (per 1000) of
    // the work, each a constant and a term per head of the group
    static constexpr double kRows[3][8] = {{2.04, 0.82, 1.47, 0.25, 0.12, 2.62, 0.52, 0.74},     // head_dim up to 64
                                           {1.36, 0.72, 2.58, 0.43, 0.29, 2.32, 1.76, 1.43},     // 128
                                           {0.12, 0.54, 4.96, 0.89, 1.88, 2.68, 3.70, 2.84}};    // 256
    // {start, step} of the chain and of 1000 waves' work; bf16 pages, then the others, each under bf16 and f32 queries
    static constexpr double kTiles[4][4][4] = {
        {{5.77, 0.72, 7.20, 1.44}, {6.34, 0.84, 10.86, 0.83}, {5.83, 1.69, 7.24, 3.68}, {6.39, 1.75, 7.77, 3.64}},        // 64
        {{7.72, 0.99, 0.00, 0.00}, {8.48, 1.17, 0.00, 7.89}, {7.69, 2.50, 0.00, 8.98}, {8.47, 3.03, 21.18, 10.35}},       // 96
        {{6.08, 3.95, 8.48, 6.65}, {6.92, 4.56, 6.41, 8.71}, {6.08, 3.95, 8.48, 6.65}, {6.92, 4.56, 6.41, 8.71}},         // 128 (f32 pages)
        {{11.29, 3.31, 9.66, 4.89}, {14.20, 7.11, 0.00, 14.55}, {4.21, 10.46, 18.65, 9.67}, {5.74, 15.17, 27.86, 11.45}}};  // 256
    const int d = a.head_dim;
    const double g = a.group <= 2 ? a.group : a.group <= 4 ? 4 : 8;
    const double *r = kRows[d <= 64 ? 0 : d <= 128 ? 1 : 2];
    const double t_rows = hypot(r[0] + r[1] * g + (r[2] + r[3] * g) * steps,
                                1e-3 * (double)wgs * (r[4] + r[5] * g + (r[6] + r[7] * g) * mean));
    const double *t = kTiles[d <= 64 ? 0 : d <= 96 ? 1 : d <= 128 ? 2 : 3]
                            [(a.dtype != AIR_KV_BF16 ? 2 : 0) + (a.q_dtype == AIR_KV_F32 ? 1 : 0)];
    const double waves = (double)held * a.group * a.n_kv_heads / 32;
    const double t_tiles = hypot(t[0] + t[1] * steps, 1e-3 * waves * (t[2] + t[3] * mean));
    return t_tiles * (a.tokens < rows + 32 ? 1.05 : 1.1) < t_rows;
}

}  // namespace airkv
