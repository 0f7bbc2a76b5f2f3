// Device-wide primitives for the binning stage on gfx950: clearing, and the records' sort, an LSD onesweep radix
// sort of (tile, depth) keys with record indices: per-digit histograms in one pass, then one scatter pass per 8-bit
// digit with in-workgroup stable ranking (wave64 ballot match), LDS reordering for contiguous writes, and decoupled
// look-back across partitions for the global offsets.
// Replaces fuchsia_radix_sort (TetMeshRendererIntersection.cpp:624-653) and its CPU std::sort fallback
// (:682-696).  Stability makes equal keys keep their input order.
#include "dtv_kernels.h"
#include "dtv_prims.h"
#include "sort_plan.h"

namespace dtv {

// ------------------------------------------------------------------------------------------------------
// Fill
__global__ void k_fill_u32(uint32_t* __restrict__ p, uint32_t v, int64_t n) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        p[i] = v;
}

void fill_u32(uint32_t* p, uint32_t v, int64_t n, hipStream_t s) {
    if (n <= 0) return;
    int64_t blocks = (n + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(k_fill_u32, dim3((unsigned)blocks), dim3(256), 0, s, p, v, n);
}

struct ClearArgs {
    ClearList list;
    BatchItem item;
    BatchItem* item_dst;
    AdjointTarget targets[kClearTargets];
    AdjointTarget* targets_dst;
    int ntargets;
};

__global__ __launch_bounds__(256) void k_clear(ClearArgs A) {
    const int64_t i0 = blockIdx.x * (int64_t)blockDim.x + threadIdx.x, step = (int64_t)gridDim.x * blockDim.x;
    for (int r = 0; r < A.list.count; r++)
        for (int64_t i = i0; i < A.list.n[r]; i += step) A.list.p[r][i] = 0u;
    if (i0 == 0 && A.item_dst != nullptr) *A.item_dst = A.item;
    if (A.targets_dst != nullptr && i0 < A.ntargets) A.targets_dst[i0] = A.targets[i0];
}

void launch_clear(const ClearList& regions, const BatchItem* item, BatchItem* item_dst, const AdjointTarget* targets,
                  int ntargets, AdjointTarget* targets_dst, hipStream_t s) {
    ClearArgs A{};
    A.list = regions;
    int64_t most = 1;
    for (int r = 0; r < regions.count; r++) most = regions.n[r] > most ? regions.n[r] : most;
    if (item != nullptr) A.item = *item;
    A.item_dst = item_dst;
    A.targets_dst = targets_dst;
    A.ntargets = ntargets;
    for (int i = 0; i < ntargets; i++) A.targets[i] = targets[i];
    int64_t blocks = (most + 1023) / 1024;  // four words a thread
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(k_clear, dim3((unsigned)blocks), dim3(256), 0, s, A);
}

// ------------------------------------------------------------------------------------------------------
// Radix sort.
// The 64-bit keys hold a tile number and a depth key (float bits); of the latter only the difference from the
// smallest one counts, about 17 bits in a view of a mesh.  The passes sort the compact key tile << dbits | (depth -
// dmin), 31 bits at 16K tiles: four passes where the raw keys' varying digits take five.  Pass 0 forms it and writes
// 32-bit keys; a compact key of more bits stays 64 bits wide until the digits sorted so far, which no later pass
// reads, can be dropped.  Record indices are not read by pass 0 either: they are the positions.
//   measured (1.57M tets at 1024 x 1024): histogram and 5 passes of 64-bit keys 468 us, and 4 passes 345 us
int sort_bits(uint32_t range) { return bits_of(range); }

int sort_max_passes(int tbits) { return plan_sort(0u, 32, tbits).passes; }

// Every lane of the wave must take part.
__device__ __forceinline__ SortPlan make_plan(const SortInput& in) {
    if (in.slots == nullptr) return plan_sort(in.dmin, in.dbits, in.tbits);
    static_assert(kBinSlots == 64, "one slot per lane");
    const BinSlot s = in.slots[lane_id()];
    const uint32_t lo = ~wave_max_u32(s.not_min), hi = wave_max_u32(s.max);
    return plan_sort(lo, hi > lo ? bits_of(hi - lo) : 0, in.tbits);
}

constexpr int kSortBlock = 256, kSortWaves = kSortBlock / 64;
// Keys per thread: many small partitions where larger ones would not fill the GPU.  Measured with 4 / 8 / 12 / 16 /
// 24 keys, us: 11K records 29 / 33 / 38 / 43 / 52, 163K 57 / 56 / 60 / 66 / 78, 510K 95 / 75 / 77 / 79 / 90, 1.0M 144 /
// 109 / 103 / 96 / 106, 10.5M 690 / 471 / 410 / 392 / 406, 81.8M 6021 / 4187 / 3601 / 3484 / 3603.
constexpr int kSortItemsSmall = 4, kSortItemsMid = 8, kSortItemsLarge = 16;
static int sort_items(int64_t n) {
    return n <= (1 << 16) ? kSortItemsSmall : n <= (5 << 17) ? kSortItemsMid : kSortItemsLarge;
}
static int64_t sort_parts(int64_t n) {
    const int64_t part = (int64_t)kSortBlock * sort_items(n);
    return (n + part - 1) / part;
}
int64_t sort_lookback_words(int64_t cap, int passes) { return 256 * (sort_parts(cap) + 1) * (int64_t)passes; }

// Histograms of every pass's digit: hist[pass][256].  One LDS histogram per wave keeps the atomics of a single heavy
// bin spread over four copies.  Also zeroes the passes' look-back words and writes the route.
__global__ __launch_bounds__(256) void k_sort_histogram(SortInput in, uint32_t* __restrict__ hist,
                                                         uint32_t* __restrict__ lookback, int64_t lookback_words,
                                                         SortRoute* __restrict__ route) {
    const int64_t n = run_count(in.cap, in.n_dev);
    const SortPlan plan = make_plan(in);
    __shared__ uint32_t s_h[4][8][256];
    for (int i = threadIdx.x; i < 4 * 8 * 256; i += 256) (&s_h[0][0][0])[i] = 0;
    const int64_t i0 = blockIdx.x * (int64_t)blockDim.x + threadIdx.x, step = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = i0; i < lookback_words; i += step) lookback[i] = 0u;
    if (i0 == 0) {
        const bool odd = plan.passes & 1;
        route->keys = reinterpret_cast<const uint32_t*>(odd ? in.keys2 : in.keys);
        route->vals = odd ? in.vals2 : in.vals;
        route->masks = reinterpret_cast<uint2*>(odd ? in.keys : in.keys2);
        route->tile_shift = plan.tile_shift();
    }
    __syncthreads();
    const int w = threadIdx.x / 64;
    const int lane = lane_id();
    for (int64_t i = i0; i < n; i += step) {
        const uint64_t k = compact_key(in.keys[i], plan);
        const uint64_t act = ballot(true);
#pragma unroll
        for (int p = 0; p < 8; p++) {
            if (p >= plan.passes) break;
            // digits shared by the whole wave (the high tile bits) are added once: 64 LDS atomics on one address
            // would serialise
            const uint32_t d = (uint32_t)(k >> (8 * p)) & 255u;
            const uint32_t d0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)d);
            if (ballot(d == d0) == act) {
                if (lane == __ffsll((unsigned long long)act) - 1) atomicAdd(&s_h[w][p][d0], (uint32_t)popc64(act));
            } else {
                atomicAdd(&s_h[w][p][d], 1u);
            }
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 256 * plan.passes; i += 256) {
        const int p = i / 256;
        const uint32_t c = s_h[0][p][i % 256] + s_h[1][p][i % 256] + s_h[2][p][i % 256] + s_h[3][p][i % 256];
        if (c) atomicAdd(&hist[i], c);
    }
}

template <int kItems, typename KeyOut>
struct SortLds {
    uint32_t part;
    uint32_t wcnt[kSortWaves][256];
    uint32_t local_start[256];
    uint32_t global_base[256];
    uint32_t tmp[kSortWaves + 1];
    KeyOut keys[kSortBlock * kItems];
    uint32_t vals[kSortBlock * kItems];
};

// One pass.  in_shift: the digit's position in the input keys; out_shift: the low bits the output keys leave out.
// kFirst: the input keys are raw, and the values are the positions.
template <int kItems, typename KeyIn, typename KeyOut, bool kFirst>
__device__ __forceinline__ void sort_pass(SortLds<kItems, KeyOut>& L, const KeyIn* __restrict__ kin,
                                          const uint32_t* __restrict__ vin, KeyOut* __restrict__ kout,
                                          uint32_t* __restrict__ vout, int64_t n, const SortPlan& plan, int in_shift,
                                          int out_shift, const uint32_t* __restrict__ hist,
                                          uint32_t* __restrict__ lookback, uint32_t* __restrict__ part_counter) {
    constexpr int kPart = kSortBlock * kItems;
    if (threadIdx.x == 0) L.part = atomicAdd(part_counter, 1u);
    for (int i = threadIdx.x; i < kSortWaves * 256; i += kSortBlock) (&L.wcnt[0][0])[i] = 0;
    // first output position of each digit
    uint32_t all;
    const uint32_t digit_start = block_exclusive_scan<kSortBlock>(hist[threadIdx.x], L.tmp, all);
    __syncthreads();
    const uint32_t part = L.part;
    const int w = threadIdx.x / 64;
    const int lane = lane_id();
    const uint64_t lt = lanemask_lt();
    const int64_t pbase = (int64_t)part * kPart;
    if (pbase >= n) return;  // (planned launches are sized for the capacity)
    const int64_t wbase = pbase + (int64_t)w * (64 * kItems);

    KeyIn key[kItems];
    uint32_t val[kItems];
    uint32_t rank[kItems];
#pragma unroll
    for (int i = 0; i < kItems; i++) {
        const int64_t idx = wbase + i * 64 + lane;
        const bool valid = idx < n;
        if constexpr (kFirst) {
            key[i] = valid ? compact_key(kin[idx], plan) : 0;
            val[i] = (uint32_t)idx;
        } else {
            key[i] = valid ? kin[idx] : 0;
            val[i] = valid ? vin[idx] : 0u;
        }
    }
    // Stable rank inside the wave: items are visited in input order (slot i, then lane).  For each slot the
    // lowest lane of every digit adds the slot's count of that digit to the wave's counter and gets the count
    // before it back; the LDS runs one wave's atomics in issue order, so the slots need not wait on each other.
    // The other lanes then take their leader's base by a lane permute.
    uint32_t info[kItems];  // rank among the slot's lanes of the same digit | leader lane << 8
#pragma unroll
    for (int i = 0; i < kItems; i++) {
        const int64_t idx = wbase + i * 64 + lane;
        const bool valid = idx < n;
        const uint32_t d = (uint32_t)(key[i] >> in_shift) & 255u;
        uint64_t peers = ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; b++) {
            const bool bit = (d >> b) & 1u;
            const uint64_t bb = ballot(bit);
            peers &= bit ? bb : ~bb;
        }
        const uint32_t below = (uint32_t)popc64(peers & lt);
        const uint32_t cnt = (uint32_t)popc64(peers);
        const int leader = peers != 0ull ? __ffsll((unsigned long long)peers) - 1 : lane;
        uint32_t base = 0u;
        if (valid && below == 0) base = atomicAdd(&L.wcnt[w][d], cnt);
        rank[i] = base;
        info[i] = below | ((uint32_t)leader << 8);
    }
#pragma unroll
    for (int i = 0; i < kItems; i++)
        rank[i] = (uint32_t)__shfl((int)rank[i], (int)(info[i] >> 8), 64) + (info[i] & 255u);
    __syncthreads();
    // Per digit (one thread each): wave offsets, block total, look-back for the global base.
    const uint32_t d = threadIdx.x;
    uint32_t run = 0;
#pragma unroll
    for (int ww = 0; ww < kSortWaves; ww++) {
        const uint32_t c = L.wcnt[ww][d];
        L.wcnt[ww][d] = run;
        run += c;
    }
    const uint32_t total_d = run;
    uint32_t* my = lookback + (int64_t)part * 256 + d;
    uint32_t excl = 0;
    if (part == 0) {
        status_store(my, kFlagInc | total_d);
    } else {
        status_store(my, kFlagAgg | total_d);
        // four partitions' words in flight at a time
        bool known = false;
        for (int64_t p = (int64_t)part - 1; p >= 0 && !known;) {
            uint32_t wv[4];
#pragma unroll
            for (int q = 0; q < 4; q++) wv[q] = p - q >= 0 ? status_load(lookback + (p - q) * 256 + d) : kFlagInc;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const uint32_t flag = wv[q] & ~kValMask;
                if (known || flag == 0u) break;
                excl += wv[q] & kValMask;
                known = flag == kFlagInc;
                p--;
            }
        }
        status_store(my, kFlagInc | (excl + total_d));
    }
    L.global_base[d] = digit_start + excl;
    uint32_t blk_total;
    const uint32_t lstart = block_exclusive_scan<kSortBlock>(total_d, L.tmp, blk_total);
    L.local_start[d] = lstart;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kItems; i++) {
        const int64_t idx = wbase + i * 64 + lane;
        if (idx < n) {
            const uint32_t dd = (uint32_t)(key[i] >> in_shift) & 255u;
            const uint32_t lp = L.local_start[dd] + L.wcnt[w][dd] + rank[i];
            // the output position travels with the item: the output key may no longer hold this digit
            L.keys[lp] = (KeyOut)(key[i] >> out_shift);
            L.vals[lp] = val[i];
        }
    }
    __syncthreads();
    const int64_t valid_n = (n - pbase) < kPart ? (n - pbase) : kPart;
    for (int j = threadIdx.x; j < valid_n; j += kSortBlock) {
        // the digit of reordered item j: the last one whose first local position is at most j
        uint32_t dd;
        const KeyOut k = L.keys[j];
        if (in_shift >= out_shift) {
            dd = (uint32_t)(k >> (in_shift - out_shift)) & 255u;
        } else {
            uint32_t lo = 0, hi = 255;
            while (lo < hi) {
                const uint32_t mid = (lo + hi + 1) >> 1;
                if (L.local_start[mid] <= (uint32_t)j) lo = mid; else hi = mid - 1;
            }
            dd = lo;
        }
        const uint32_t dest = L.global_base[dd] + ((uint32_t)j - L.local_start[dd]);
        kout[dest] = k;
        vout[dest] = L.vals[j];
    }
}

// kWide: the host does not know whether the pass reads or writes 64-bit keys (planned), or it does and they are;
// else the keys are 32 bits, raw 64-bit ones into pass 0.
template <int kItems, bool kWide, bool kFirst>
__global__ __launch_bounds__(kSortBlock) void k_sort_pass(SortInput in, int pass, const uint32_t* __restrict__ hist,
                                                          uint32_t* __restrict__ lookback,
                                                          uint32_t* __restrict__ part_counter) {
    const int64_t n = run_count(in.cap, in.n_dev);
    const SortPlan plan = make_plan(in);
    if (pass >= plan.passes) return;
    const bool odd = pass & 1;
    uint64_t* kin = odd ? in.keys2 : in.keys;
    uint64_t* kout = odd ? in.keys : in.keys2;
    const uint32_t* vin = odd ? in.vals2 : in.vals;
    uint32_t* vout = odd ? in.vals : in.vals2;
    uint32_t* kout32 = reinterpret_cast<uint32_t*>(kout);
    if constexpr (!kWide) {
        __shared__ SortLds<kItems, uint32_t> L;
        if constexpr (kFirst)
            sort_pass<kItems, uint64_t, uint32_t, true>(L, kin, vin, kout32, vout, n, plan, 0, plan.drop, hist,
                                                        lookback, part_counter);
        else
            sort_pass<kItems, uint32_t, uint32_t, false>(L, reinterpret_cast<const uint32_t*>(kin), vin, kout32, vout,
                                                         n, plan, 8 * pass - plan.drop, 0, hist, lookback,
                                                         part_counter);
    } else {
        __shared__ union {
            SortLds<kItems, uint64_t> wide;
            SortLds<kItems, uint32_t> narrow;
        } L;
        const int lw = plan.last_wide();
        if (pass > lw)
            sort_pass<kItems, uint32_t, uint32_t, false>(L.narrow, reinterpret_cast<const uint32_t*>(kin), vin, kout32,
                                                         vout, n, plan, 8 * pass - plan.drop, 0, hist, lookback,
                                                         part_counter);
        else if (pass == lw)
            sort_pass<kItems, uint64_t, uint32_t, kFirst>(L.narrow, kin, vin, kout32, vout, n, plan, 8 * pass,
                                                          plan.drop, hist, lookback, part_counter);
        else
            sort_pass<kItems, uint64_t, uint64_t, kFirst>(L.wide, kin, vin, kout, vout, n, plan, 8 * pass, 0, hist,
                                                          lookback, part_counter);
    }
}

template <int kItems>
static void launch_pass(const SortInput& in, int pass, bool wide, int64_t parts, const uint32_t* hist,
                        uint32_t* lookback, uint32_t* counter, hipStream_t s) {
    const dim3 g((unsigned)parts), b(kSortBlock);
    if (wide && pass == 0)
        hipLaunchKernelGGL((k_sort_pass<kItems, true, true>), g, b, 0, s, in, pass, hist, lookback, counter);
    else if (wide)
        hipLaunchKernelGGL((k_sort_pass<kItems, true, false>), g, b, 0, s, in, pass, hist, lookback, counter);
    else if (pass == 0)
        hipLaunchKernelGGL((k_sort_pass<kItems, false, true>), g, b, 0, s, in, pass, hist, lookback, counter);
    else
        hipLaunchKernelGGL((k_sort_pass<kItems, false, false>), g, b, 0, s, in, pass, hist, lookback, counter);
}

int sort_records(const SortInput& in, uint32_t* hist, uint32_t* counters, uint32_t* lookback, SortRoute* route,
                 hipStream_t s) {
    if (in.cap <= 0) return 0;
    const bool planned = in.slots != nullptr;
    const SortPlan plan = plan_sort(in.dmin, planned ? 32 : in.dbits, in.tbits);  // planned: the most passes
    const int last_wide = plan.last_wide();
    const int64_t parts = sort_parts(in.cap);
    const int items = sort_items(in.cap);
    const int64_t words = 256 * parts;
    int64_t hblocks = (in.cap + 2047) / 2048;  // a block's 256 sums per pass go out as global atomics
    if (hblocks > 1024) hblocks = 1024;
    hipLaunchKernelGGL(k_sort_histogram, dim3((unsigned)hblocks), dim3(256), 0, s, in, hist, lookback,
                       words * plan.passes, route);
    for (int p = 0; p < plan.passes; p++) {
        // 64-bit keys beyond pass 0's input: when planned, up to the last pass that may read them
        const bool wide = planned ? p <= last_wide : plan.drop > 8 && p <= last_wide;
        uint32_t* lb = lookback + words * p;
        if (items == kSortItemsSmall)
            launch_pass<kSortItemsSmall>(in, p, wide, parts, hist + 256 * p, lb, counters + p, s);
        else if (items == kSortItemsMid)
            launch_pass<kSortItemsMid>(in, p, wide, parts, hist + 256 * p, lb, counters + p, s);
        else
            launch_pass<kSortItemsLarge>(in, p, wide, parts, hist + 256 * p, lb, counters + p, s);
    }
    return plan.passes;
}

}  // namespace dtv
