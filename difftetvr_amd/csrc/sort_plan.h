// Arithmetic of the record sort's compact keys, for the device and for host code of any compiler.
#pragma once
#include <stdint.h>

#ifdef __HIPCC__
#define DTV_HOST_DEVICE __host__ __device__
#else
#define DTV_HOST_DEVICE
#endif

namespace dtv {

struct SortPlan {
    uint32_t dmin;
    int dbits, total;  // bits of the depth difference and of the compact key
    int passes;
    int drop;          // low bits the 32-bit keys leave out
    DTV_HOST_DEVICE int last_wide() const { return drop > 0 ? drop / 8 - 1 : 0; }  // last pass that reads 64 bits
    DTV_HOST_DEVICE uint32_t tile_shift() const { return (uint32_t)(dbits - drop); }  // of the 32-bit keys: 0 to 32
};

DTV_HOST_DEVICE inline int bits_of(uint32_t x) { return x == 0u ? 0 : 32 - __builtin_clz(x); }

DTV_HOST_DEVICE inline SortPlan plan_sort(uint32_t dmin, int dbits, int tbits) {
    SortPlan p;
    p.dmin = dmin;
    p.dbits = tbits > 24 ? 32 : dbits;  // the dropped digits then never reach the tile bits
    p.total = p.dbits + tbits;
    p.passes = p.total <= 8 ? 1 : (p.total + 7) / 8;
    p.drop = p.total > 32 ? 8 * ((p.total - 32 + 7) / 8) : 0;
    return p;
}

DTV_HOST_DEVICE inline uint64_t compact_key(uint64_t k, const SortPlan& p) {
    return ((k >> 32) << p.dbits) | (uint64_t)((uint32_t)k - p.dmin);
}

// Tile of a sorted 32-bit key.  The shift is 32 where a view of a single tile holds depth keys on either side of the
// sign bit (a face at the near plane whose centroid rounds below 0): the key is all depth then, and a 32-bit shift by
// 32 would not give tile 0.
DTV_HOST_DEVICE inline uint32_t tile_of_key(uint32_t key, uint32_t tile_shift) {
    return (uint32_t)((uint64_t)key >> tile_shift);
}

}  // namespace dtv
