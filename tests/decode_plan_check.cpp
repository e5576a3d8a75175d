// Checks decode_plan.hpp against a walk over the pieces it describes: every cut
// piece of a launch gets a row of its own inside the planned slots, the
// workspace stays within its bound, and the plan uses the GPU's waves.
// Prints "<cases> cases, <n> wrong".
#include <algorithm>
#include <cstdio>
#include <random>
#include <vector>

#include "kernels/decode_plan.hpp"

using namespace airkv;

static long cases = 0, wrong = 0;
static void check(bool ok, const char *what, long long a = 0, long long b = 0, long long c = 0) {
    if (!ok && wrong++ < 20) std::printf("wrong: %s (%lld, %lld, %lld)\n", what, a, b, c);
}

// The pieces of sequences of these tiles in slices as the kernels cut them (full
// 0: the f32-precision one).
static void walk(const std::vector<int> &tiles, int slices, int simd, int full, int max_splits) {
    ++cases;
    long total = 0;
    int tmax = 0;
    for (int t : tiles) { total += t; tmax = std::max(tmax, t); }
    if (!total) return;
    const int chunk = full ? slice_chunk((int)total, slices, simd, full, tmax, max_splits)
                           : shared_chunk((int)total, slices, simd, tmax, max_splits);
    check(chunk >= 1 && (long)chunk * slices >= total, "the slices cover every tile", total, slices, chunk);
    const long rows = part_rows(slices, (long)tiles.size());
    long start = 0, last = -1;
    for (int b = 0; b < (int)tiles.size(); start += tiles[b], ++b) {
        if (!tiles[b]) continue;
        const int w0 = (int)(start / chunk), w1 = (int)((start + tiles[b] - 1) / chunk);
        check(w1 - w0 + 1 <= max_splits * (full ? 1 : kSharing), "pieces per sequence", w1 - w0 + 1, max_splits);
        if (w0 == w1) continue;
        for (int w = w0; w <= w1; ++w) {
            const int row = part_row(w, b, w == w0);
            check(row > last && row < rows, "a row of its own inside the slots", row, last, rows);
            check((w == w0) == (start >= (long)w * chunk), "the kernel's test of a first piece", w, w0);
            last = row;
        }
    }
}

// The same where every sequence has `pieces` slices of its own.
static void walk_own(const std::vector<int> &tiles, int pieces) {
    ++cases;
    for (int t : tiles) {
        if (!t) continue;
        const int step = piece_tiles(t, pieces), n = (t + step - 1) / step;
        check(n >= 1 && n <= pieces && (long)step * pieces >= t, "a sequence's own slices cover it", t, pieces, step);
    }
}

int main() {
    std::mt19937 rng(5);
    auto in = [&](int lo, int hi) { return lo + (int)(rng() % (unsigned)(hi - lo + 1)); };
    for (int i = 0; i < 20000; ++i) {
        const int B = i % 3 ? in(1, 40) : in(1, 1500), most = in(0, 3) ? in(1, 9) : in(1, 400);
        std::vector<int> tiles(B);
        for (int &t : tiles) t = in(0, most);
        const int splits = in(0, 2) ? 64 : in(1, 256);
        if (splits > 1) walk(tiles, in(1, std::min(4096, B * splits)), in(1, 1024), 0, splits);
        walk(tiles, in(1, std::min(4096, B * splits)), in(1, 1024), in(1, 4), splits);
        walk_own(tiles, in(1, 4));
    }
    // the widest launches: tile counts up to the plan's bound
    for (int64_t blocks : {(int64_t)INT32_MAX, (int64_t)(1 << 27), (int64_t)(1 << 26) - 1, (int64_t)(1 << 20) + 7, (int64_t)524288})
        for (int batch : {1, 3, 15, 16, 31, 4096}) {
            ++cases;
            const DecodeF32Plan p = plan_f32(8, 8, 64, 16, batch, blocks, 64, 4096, 3072);
            const int64_t tiles = std::min<int64_t>(blocks, ((int64_t)INT32_MAX + 15) / 16), total = p.batch * tiles;
            check(p.batch >= 1 && total + 65536 <= INT32_MAX, "tiles of a launch", total, p.batch, blocks);
            for (int slices : {1, 384, 16384}) {
                const int c = shared_chunk((int)total, slices, 128, (int)tiles, 64);
                check(c >= 1 && (int64_t)c * slices >= total, "slices of a wide launch", c, slices, total);
                const int d = slice_chunk(INT32_MAX, slices, 128, 4, (int)tiles, 64);
                check(d >= 1 && (int64_t)d * slices >= INT32_MAX, "slices of the widest", d, slices);
            }
        }
    // slices of a plan: waves of a 256-CU GPU, the cap or a row per (sequence, 256 tokens)
    const size_t cap = kWsBytes;
    for (int nkv : {1, 2, 4, 8, 16})
        for (int group : {1, 4, 8, 16, 32, 71})
            for (int d : {32, 64, 96, 128, 256})
                for (int batch : {1, 4, 64, 253, 300, 380, 512, 1024, 2048, 4096, 5000})
                    for (int blocks : {1, 4, 16, 64, 8192})
                        for (int splits : {1, 2, 64, 256}) {
                            ++cases;
                            const int64_t nq = nkv * group, per = nkv * ((group + 15) / 16), row = nq * (d + 2) * 4;
                            const DecodeF32Plan p = plan_f32(nq, per, d, 16, batch, blocks, splits, 4096, 3072);
                            const int64_t parts = std::min<int64_t>(splits, (blocks + 15) / 16);
                            check(p.ws_bytes <= std::max<size_t>(cap, (size_t)row * p.batch * parts), "workspace", (long long)p.ws_bytes, row, batch);
                            check(p.slices_qf32 <= p.slices && p.slices_qf32 >= 1, "slices");
                            const int64_t fit = std::max<int64_t>(1, ((int64_t)cap - 20000) / row);
                            if (splits == 1) {                   // every sequence its own slices, as many as its partition's waves
                                check(p.slices == p.batch * p.seq_pieces && p.slots >= (p.seq_pieces > 1 ? p.slices : 1), "own slots");
                                check(p.seq_pieces <= kSharing && p.seq_pieces >= std::min<int64_t>(std::min<int64_t>(kSharing, (blocks + 1) / 2), fit / p.batch),
                                      "own slices", p.seq_pieces, blocks, fit);
                                continue;
                            }
                            check(!p.seq_pieces && p.slots == part_rows(p.slices, p.batch), "slots");
                            // half the partial rows of the cap at least, unless the waves or the splits are fewer
                            const int64_t want = std::min(std::min<int64_t>((4096 + per - 1) / per, p.batch * std::min(splits * kSharing, blocks)),
                                                          std::max<int64_t>(1, fit / 2));
                            check(p.slices >= want, "slices of a wide batch", p.slices, want, batch);
                        }
    std::printf("%ld cases, %ld wrong\n", cases, wrong);
    return wrong != 0;
}
