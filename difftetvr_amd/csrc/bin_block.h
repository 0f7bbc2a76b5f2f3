// The part of binning that the tile and the Projection renderer share: one workgroup turns the screen triangles of
// 256 tets into (tile, face) records, in order, at their place in the batch's record list.
//
// A thread per tet would project and then walk its faces' tiles alone; faces cover between none and thousands of
// tiles, so most lanes would wait.  Here the workgroup lists its screen triangles in LDS, and its threads then
// share the (face, tile) candidates evenly: candidate c belongs to the face whose range of candidates holds c.  A
// candidate becomes a record when the face covers a pixel centre of the tile (exact 8x8 coverage, part of the
// record).  The workgroup's place in the list comes from a decoupled look-back over the workgroups before it, so
// one pass projects every tet once, writes the records once, and keeps (tet, face, tile) order.
//   measured (1.57M tets at 1024 x 1024): counting, scan, emission and the gather of the sorted records, each
//   projecting again, 494 us; this pass 294 us, and 9% of the records (no pixel covered) are gone.  It is bound by
//   the VALU (coverage) and by the latency of its phases.
#pragma once
#include "dtv_kernels.h"
#include "dtv_prims.h"
#include "raster.h"

namespace dtv {

constexpr int kBinBlock = 256;   // threads per workgroup
constexpr int kBinUnit = 256;    // tets per block of the batch's block grid
constexpr int kBinKeep = 8;      // rounds of 256 candidates whose coverage stays in registers between the sweeps

constexpr uint32_t kBinSearch = 0xFFFFu;  // owner: found by bisection
constexpr uint32_t kBinOwnMost = 32;      // candidates a thread lists for one face

// Faces refer to their tet's screen vertices, so that five workgroups fit in a CU's LDS.
// kTets tets per workgroup: 256 (a thread per tet), or 64, where a mesh of few tets or of large ones leaves too few
// candidates in flight (launch_bin).
template <int kTets>
struct BinLds {
    static constexpr int kFaces = 4 * kTets;   // most faces (a flat tet may show all four)
    int32_t X[5][kTets], Y[5][kTets];  // per tet: fixed-point screen vertices (Projection: five)
    uint32_t key[kFaces];                   // depth key
    uint32_t place[kFaces];                 // first tile x | y << 11, tet of the block << 22, face << 30
    uint32_t shape[kFaces];                 // tiles per row of the bounding box | record bits << 12 (9 bits)
                                               // | vertex slots, oriented to positive area << 21 (3 bits each)
    uint32_t first[kFaces + 1];             // candidates before the face
    alignas(4) uint16_t owner[kBinBlock * kBinKeep];  // face of each of the first candidates, or kBinSearch
    uint32_t tmp[kBinBlock / 64 + 1];
    uint32_t cnt[kBinKeep * (kBinBlock / 64)];
    uint32_t extra, part;
    uint64_t base;
};

// Ticket of this workgroup: the kTets tets it bins.  Taken in order, so every earlier block is already running
// when a later one waits for its count.
template <int kTets>
__device__ __forceinline__ uint32_t bin_ticket(BinLds<kTets>& L, ViewScratch* sm) {
    if (threadIdx.x == 0) {
        L.part = atomicAdd(&sm->ticket, 1u);
        L.extra = 0u;
    }
    __syncthreads();
    return L.part;
}

// Fixed-point screen vertex `slot` of this thread's tet, from its NDC x and y.
template <int kTets>
__device__ __forceinline__ void bin_vertex(const ViewUniforms& U, BinLds<kTets>& L, int slot, float nx, float ny) {
    const float hw = 0.5f * (float)U.width, hh = 0.5f * (float)U.height;
    const float xf = nx * hw + hw, yf = ny * hh + hh;
    L.X[slot][threadIdx.x] = (int32_t)rintf(xf * 256.0f);
    L.Y[slot][threadIdx.x] = (int32_t)rintf(yf * 256.0f);
}

// Lists the triangle of this thread's tet with vertex slots a, b, c as entry e; face: 2 bits of the record id,
// extra: 9 bits for the record.  Returns the number of candidate tiles.
template <int kTets>
__device__ __forceinline__ uint32_t bin_entry(const ViewUniforms& U, BinLds<kTets>& L, uint32_t e, uint32_t face,
                                              int a, int b, int c, uint32_t key, uint32_t extra) {
    const int t = threadIdx.x;
    ScreenTri S;
    S.X[0] = L.X[a][t];
    S.Y[0] = L.Y[a][t];
    S.X[1] = L.X[b][t];
    S.Y[1] = L.Y[b][t];
    S.X[2] = L.X[c][t];
    S.Y[2] = L.Y[c][t];
    S.area2 = (int64_t)(S.X[1] - S.X[0]) * (int64_t)(S.Y[2] - S.Y[0]) -
              (int64_t)(S.Y[1] - S.Y[0]) * (int64_t)(S.X[2] - S.X[0]);
    const bool turned = S.area2 < 0;  // (the bounding box does not depend on the orientation)
    const FaceBins bins = screen_bins(U, S);
    const uint32_t w = bins.tx0 > bins.tx1 ? 0u : (uint32_t)(bins.tx1 - bins.tx0 + 1);
    const uint32_t n = bins.ty0 > bins.ty1 ? 0u : w * (uint32_t)(bins.ty1 - bins.ty0 + 1);
    L.key[e] = key;
    L.place[e] = (uint32_t)max(bins.tx0, 0) | ((uint32_t)max(bins.ty0, 0) << 11) | ((uint32_t)t << 22) | (face << 30);
    L.shape[e] = w | (extra << 12) | ((uint32_t)(a | ((turned ? c : b) << 3) | ((turned ? b : c) << 6)) << 21);
    L.first[e] = n;
    return n;
}

struct BinCandidate {
    uint32_t face, tx, ty;
    uint64_t mask;  // 8x8 tiles: the covered pixels (larger tiles: 0, tested by the renderer)
    bool keep;
};

template <int kTets>
__device__ __forceinline__ BinCandidate bin_candidate(const ViewUniforms& U, const BinLds<kTets>& L,
                                                      uint32_t nfaces, uint32_t c) {
    uint32_t lo = c < (uint32_t)(kBinBlock * kBinKeep) ? L.owner[c] : kBinSearch;
    if (lo == kBinSearch) {
        lo = 0;
        uint32_t hi = nfaces - 1u;
        while (lo < hi) {
            const uint32_t mid = (lo + hi + 1u) >> 1;
            if (L.first[mid] <= c) lo = mid; else hi = mid - 1u;
        }
    }
    BinCandidate r;
    r.face = lo;
    const uint32_t shape = L.shape[lo], place = L.place[lo];
    const uint32_t w = shape & 0xFFFu, k = c - L.first[lo], tet = (place >> 22) & 255u;
    // k / w: exact below 2^12 by the reciprocal (its error stays far below the quotient's distance 1 / 2w to an
    // integer)
    const uint32_t row = k < 4096u ? (uint32_t)(((float)k + 0.5f) * __builtin_amdgcn_rcpf((float)w)) : k / w;
    r.tx = (place & 0x7FFu) + (k - row * w);
    r.ty = ((place >> 11) & 0x7FFu) + row;
    ScreenTri S;
#pragma unroll
    for (int q = 0; q < 3; q++) {
        const uint32_t v = (shape >> (21 + 3 * q)) & 7u;
        S.X[q] = L.X[v][tet];
        S.Y[q] = L.Y[v][tet];
    }
    S.area2 = 1;  // not read by the tests below
    r.mask = 0ull;
    if (U.tile_shift == 3) {
        r.mask = tile_coverage(S, (int)r.tx, (int)r.ty, U.width, U.height);
        r.keep = r.mask != 0ull;
    } else {
        const uint32_t all = L.first[lo + 1u] - L.first[lo];
        r.keep = all > (uint32_t)kMaxTestedTiles || tile_may_cover(S, (int)r.tx, (int)r.ty, U.tile_shift);
    }
    return r;
}

// The listed faces' records.  nparts: workgroups of the launch.  kWide: two uint4 per record, {tet vertex indices},
// {id, mask low, high, extra}; else the second alone.
template <bool kWide, int kTets>
__device__ __forceinline__ void bin_emit(const BatchItem& B, BinLds<kTets>& L, uint32_t nfaces, uint32_t part,
                                         uint32_t nparts, const BinOut& out) {
    constexpr int kFaces = BinLds<kTets>::kFaces;
    const ViewUniforms& U = B.U;
    const int t = threadIdx.x, w = t >> 6;
    const int lane = lane_id();
    const uint64_t lt = lanemask_lt();
    for (int i = t; i < kBinBlock * kBinKeep / 2; i += kBinBlock) reinterpret_cast<uint32_t*>(L.owner)[i] = ~0u;
    __syncthreads();
    // candidates before each face
    uint32_t C;
    {
        uint32_t v[kFaces / kBinBlock], sum = 0;
#pragma unroll
        for (int i = 0; i < kFaces / kBinBlock; i++) {
            const uint32_t e = (uint32_t)(t * (kFaces / kBinBlock) + i);
            v[i] = e < nfaces ? L.first[e] : 0u;
            sum += v[i];
        }
        uint32_t run = block_exclusive_scan<kBinBlock>(sum, L.tmp, C);
#pragma unroll
        for (int i = 0; i < kFaces / kBinBlock; i++) {
            const uint32_t e = (uint32_t)(t * (kFaces / kBinBlock) + i);
            if (e < nfaces) L.first[e] = run;
            // the face's candidates know their owner, unless they are too many for one thread to list
            const uint32_t end = min(run + v[i], (uint32_t)(kBinBlock * kBinKeep));
            const bool listed = v[i] <= kBinOwnMost;
            if (listed)
                for (uint32_t c = run; c < end; c++) L.owner[c] = (uint16_t)e;
            run += v[i];
        }
        if (t == 0) L.first[nfaces] = C;
    }
    __syncthreads();
    // first sweep: coverage and counts
    uint64_t mask[kBinKeep];
    uint32_t face[kBinKeep], tile[kBinKeep], kept = 0u;
#pragma unroll
    for (int k = 0; k < kBinKeep; k++) {
        mask[k] = 0ull;
        face[k] = tile[k] = 0u;
        const uint32_t c = (uint32_t)(kBinBlock * k + t);
        if (c < C) {
            const BinCandidate r = bin_candidate(U, L, nfaces, c);
            mask[k] = r.mask;
            face[k] = r.face;
            tile[k] = r.ty * (uint32_t)U.tiles_x + r.tx;
            kept |= (r.keep ? 1u : 0u) << k;
        }
        const uint64_t m = ballot((kept >> k) & 1u);
        if (lane == 0) L.cnt[k * (kBinBlock / 64) + w] = (uint32_t)popc64(m);
    }
    if (C > (uint32_t)(kBinBlock * kBinKeep)) {
        uint32_t n = 0;
        for (uint32_t c = (uint32_t)(kBinBlock * kBinKeep + t); c < C; c += kBinBlock)
            n += bin_candidate(U, L, nfaces, c).keep ? 1u : 0u;
        atomicAdd(&L.extra, n);
    }
    __syncthreads();
    if (w == 0) {
        constexpr int kCnt = kBinKeep * (kBinBlock / 64);
        static_assert(kCnt <= 64, "one wave scans the counts");
        const uint32_t v = lane < kCnt ? L.cnt[lane] : 0u;
        const uint32_t inc = wave_inclusive_scan(v);
        if (lane < kCnt) L.cnt[lane] = inc - v;
        const uint32_t kept_all = (uint32_t)__builtin_amdgcn_readlane((int)inc, 63);
        if (lane == 0) L.tmp[0] = kept_all;
        const uint64_t total = (uint64_t)kept_all + L.extra;
        const uint64_t before = lookback_sum(out.status, part, total);
        if (lane == 0) {
            L.base = before;
            if (part == nparts - 1u) out.scratch->total = before + total;
        }
    }
    __syncthreads();
    // second sweep: the records
    const uint64_t base = L.base;
    auto put = [&](uint64_t o, uint32_t f, uint32_t tl, uint64_t m) {
        if (o >= out.cap) {
            out.scratch->overflow = 1u;
            return;
        }
        out.keys[o] = ((uint64_t)(B.tile0 + tl) << 32) | (uint64_t)L.key[f];
        const uint32_t place = L.place[f];
        const uint32_t id = 4u * (part * kTets - B.block0 * kBinUnit + ((place >> 22) & 255u)) + (place >> 30);
        const uint4 rec = make_uint4(id, (uint32_t)m, (uint32_t)(m >> 32), (L.shape[f] >> 12) & 0x1FFu);
        if constexpr (kWide) {
            out.recs[2 * o] = *reinterpret_cast<const uint4*>(B.cells + 4 * (int64_t)(id >> 2));
            out.recs[2 * o + 1] = rec;
        } else {
            out.recs[o] = rec;
        }
    };
#pragma unroll
    for (int k = 0; k < kBinKeep; k++) {
        const bool keep = (kept >> k) & 1u;
        const uint64_t m = ballot(keep);
        if (keep) put(base + L.cnt[k * (kBinBlock / 64) + w] + (uint32_t)popc64(m & lt), face[k], tile[k], mask[k]);
    }
    uint64_t run = base + L.tmp[0];
    for (uint32_t c0 = kBinBlock * kBinKeep; c0 < C; c0 += kBinBlock) {
        BinCandidate r;
        r.keep = false;
        if (c0 + t < C) r = bin_candidate(U, L, nfaces, c0 + t);
        const uint64_t m = ballot(r.keep);
        __syncthreads();
        if (lane == 0) L.cnt[w] = (uint32_t)popc64(m);
        __syncthreads();
        uint32_t before = 0, all = 0;
        for (int q = 0; q < kBinBlock / 64; q++) {
            before += q < w ? L.cnt[q] : 0u;
            all += L.cnt[q];
        }
        if (r.keep)
            put(run + before + (uint32_t)popc64(m & lt), r.face, r.ty * (uint32_t)U.tiles_x + r.tx, r.mask);
        run += all;
    }
}

// The block's triangle count and the range of its depth keys (over faces with candidate tiles), into one of 64
// slots: one address for every workgroup would serialise.
__device__ __forceinline__ void bin_stats(ViewScratch* sm, uint32_t part, uint32_t ntri, uint32_t kmin,
                                          uint32_t kmax) {
    const uint32_t n = wave_sum_u32(ntri), lo = wave_max_u32(~kmin), hi = wave_max_u32(kmax);
    if (lane_id() == 0) {
        BinSlot* s = &sm->slots[part & (kBinSlots - 1)];
        if (n) atomicAdd(&s->tris, n);
        if (lo) atomicMax(&s->not_min, lo);
        if (hi) atomicMax(&s->max, hi);
    }
}

}  // namespace dtv
