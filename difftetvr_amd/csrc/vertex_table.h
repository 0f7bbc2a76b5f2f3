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

// The adjoint's flush: up to 128 vertex slots a batch (32 records), about 18 distinct vertices where tets share them.  Where
// every tet has its own the table overflows, and a slot that finds no entry issues its own atomics; probed to the end
// the full table cost it 96 dependent compare-and-swaps.  Adjoint, us, with 160 entries that hold every slot / 96 probed
// to the end / 96 with 4 / 8 / 16 probes, own vertices: 1,296 tets at 64^2 42 / 58 / 39 / 38 / 40, 24,576 at 512^2 561 /
// 605 / 593 / 530 / 526, 1.57M at 1024^2 6536 / 6450 / 5777 / 5792 / 5911, ball of 2,000 points at 512^2 443 / 492 / 489 /
// 447 / 438; with shared vertices 4, 8 and 16 differ by less than 3 %, 8 is best.
constexpr int kFlushTab = 96, kFlushProbes = 8;

}  // namespace dtv
