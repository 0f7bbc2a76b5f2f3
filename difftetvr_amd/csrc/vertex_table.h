// A hash table of vertex ids with a bounded number of probes, for the device and for host code of any compiler.
#pragma once
#include <stdint.h>

#ifndef DTV_HOST_DEVICE
#ifdef __HIPCC__
#define DTV_HOST_DEVICE __host__ __device__
#else
#define DTV_HOST_DEVICE
#endif
#endif

namespace dtv {

// The entry of vertex v among kTab (-1: the kProbes entries it may take hold other vertices); created: v was not there
// before.  cas(e, v) writes v to entry e if that is free (-1) and returns what it held.
template <int kTab, int kProbes, typename Cas>
DTV_HOST_DEVICE inline int vertex_entry(int32_t v, bool& created, Cas cas) {
    static_assert(kTab <= 256 && kProbes <= kTab, "the hash has 8 bits");
    created = false;
    // multiplicative hash -> [0, kTab): consecutive ids (tets with vertices of their own) spread evenly
    int e = (int)(((uint32_t)v * 2654435761u) >> 24) * kTab >> 8;
    for (int probe = 0; probe < kProbes; probe++) {
        const int32_t old = cas(e, v);
        if (old == -1 || old == v) {
            created = old == -1;
            return e;
        }
        e = e + 1 == kTab ? 0 : e + 1;
    }
    return -1;
}

// The adjoint's flush: up to 128 vertex slots a batch (32 records), about 18 distinct vertices where tets share them.
// Where every tet has its own the table overflows, and a slot that finds no entry issues its own atomics; probed to the
// end the full table cost it 96 dependent compare-and-swaps.  Adjoint, us, with 160 entries that hold every slot / 96
// probed to the end / 96 with 4 / 8 / 16 probes, own vertices: 1,296 tets at 64^2 42 / 58 / 39 / 38 / 40, 24,576 at
// 512^2 561 / 605 / 593 / 530 / 526, 1.57M at 1024^2 6536 / 6450 / 5777 / 5792 / 5911, ball of 2,000 points at 512^2
// 443 / 492 / 489 / 447 / 438; with shared vertices 4, 8 and 16 differ by less than 3 %, 8 is best.
constexpr int kFlushTab = 96, kFlushProbes = 8;

// As vertex_entry, for the regulariser's larger tables: sixteen consecutive ids lie in consecutive entries, so that the
// flush's lanes add to consecutive addresses; the probes step from group to group.
template <int kTab, int kProbes, typename Cas>
DTV_HOST_DEVICE inline int grouped_entry(int32_t v, Cas cas) {
    const uint32_t h = ((uint32_t)v >> 4) * 2654435761u;
    int e = (int)((h >> 16) & (uint32_t)(kTab / 16 - 1)) * 16 + (v & 15);
    for (int p = 0; p < kProbes; p++) {
        const int32_t old = cas(e, v);
        if (old == -1 || old == v) return e;
        e = (e + 16) & (kTab - 1);
    }
    return -1;
}

// The regulariser's workgroup: threads, and consecutive tets that each takes.
struct RegRange {
    int threads, per;
};

// A range of more tets has fewer distinct vertices a tet (of a 64^3 cube grid 2,048 tets have 0.40, 1,024 0.47), so it
// issues fewer atomics, while a thread with more tets has a longer chain of table searches, and a table that the
// vertices of its tets overfill merges nothing (it holds 4 a thread).  So: a tet a thread for small meshes and for
// those whose tets share few vertices (two a tet on average, or more), else two, and four in larger workgroups where
// those still give every CU one.
// Measured, us, one atomic per value / 128 x 1 / 256 x 2 / 512 x 4 threads x tets: cube grids of 10,368 tets 12 / 4.0 /
// 5.7 / 8.6, 82,944 43 / 5.2 / 5.7 / 8.7, 384,000 179 / 14 / 8.6 / 11, 1.57M 742 / 48 / 25 / 24; Delaunay balls of
// 12,666 tets 18 / 5.0 / 7.9 / 12, 400,374 272 / 29 / 32 / 42; 24,576 tets of a grid in random order 20 / 10 / 14 / 20;
// tets with vertices of their own, 384 3.7 / 4.5 / 7.4 / 12, 10,368 6.8 / 4.7 / 8.6 / 21, 1.57M 714 / 105 / 519 / 722.
inline RegRange regularizer_range(int64_t T, int64_t V) {
    if (T < (1 << 17) || V >= 2 * T) return {128, 1};
    return T < (1 << 19) ? RegRange{256, 2} : RegRange{512, 4};
}
constexpr int kRegProbes = 4;

}  // namespace dtv
