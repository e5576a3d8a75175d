// Key tiles of the f32-precision prefill, in host and device code, so that the
// arithmetic can be checked on the CPU (tests/prefill_tiles_check.cpp).  A
// sequence holds up to 2^31 - 1 keys and the loads run up to three tiles past its
// last, so the keys of a tile are numbered in unsigned 32 bits.
#pragma once

#include <stdint.h>

#ifdef __HIPCC__
#define AIRKV_HD __host__ __device__
#else
#define AIRKV_HD
#endif

namespace airkv {

// Tiles of kt keys (a power of two) that hold `keys` keys.
AIRKV_HD inline int key_tiles(int keys, int kt) { return (int)(((uint32_t)keys + (uint32_t)kt - 1) / (uint32_t)kt); }

// Row r of tile t.
AIRKV_HD inline uint32_t tile_key(int t, int kt, int r) { return (uint32_t)t * (uint32_t)kt + (uint32_t)r; }

// A key whose table entry row r of tile t reads: itself, or past `keys` the last.
AIRKV_HD inline uint32_t entry_key(int t, int kt, int r, int keys) {
    const uint32_t k = tile_key(t, kt, r);
    return k < (uint32_t)keys ? k : (uint32_t)keys - 1;
}

// The last of the wave's 32-row groups that starts below `keys`, as rows of tile t.
AIRKV_HD inline int tile_rows(int t, int kt, int keys) {
    return (int)(((uint32_t)keys - tile_key(t, kt, 0) + 31) & ~31u);
}

}  // namespace airkv
