// Checks prefill_tiles.hpp against 64-bit arithmetic: sequences of up to 2^31 - 1
// keys, every row of the first and last tiles and of the three past the last that
// the loads look at.  Prints "<cases> cases, <n> wrong".
#include <cstdint>
#include <cstdio>
#include <initializer_list>

#include "kernels/prefill_tiles.hpp"

using namespace airkv;

int main() {
    long cases = 0, wrong = 0;
    const int64_t top = 2147483647;
    for (int kt : {32, 64, 128})
        for (int64_t span : {(int64_t)1, top - 700})
            for (int64_t keys = span; keys <= (span == 1 ? 700 : top); ++keys) {
                const int64_t nt = (keys + kt - 1) / kt;
                ++cases;
                if (key_tiles((int)keys, kt) != nt) ++wrong;
                for (int64_t t = nt > 2 ? nt - 2 : 0; t < nt + 3; ++t) {
                    if (t < nt && tile_rows((int)t, kt, (int)keys) != (keys - t * kt + 31) / 32 * 32) ++wrong;
                    for (int r = 0; r < kt; ++r) {
                        const int64_t k = t * kt + r;
                        if (tile_key((int)t, kt, r) != (uint64_t)k) ++wrong;
                        if ((tile_key((int)t, kt, r) < (uint32_t)keys) != (k < keys)) ++wrong;
                        if (entry_key((int)t, kt, r, (int)keys) != (uint64_t)(k < keys ? k : keys - 1)) ++wrong;
                    }
                }
            }
    std::printf("%ld cases, %ld wrong\n", cases, wrong);
    return wrong != 0;
}
