// Per-view tet projection, front-face culling and screen-tile binning on gfx950.
//
// Replaces GenerateTrianglesIntersect.glsl:74-132 (per-tet projection + front faces, one atomic append each),
// ComputeTriangleDepths.glsl:72-110 (centroid-depth keys) and the rasteriser's fragment generation.  Each front
// face becomes one (tile, face) record per 8x8 screen tile with a pixel centre it covers, keyed by
// (tile << 32 | depth-key bits), with the exact 64-bit coverage mask of the tile (bin_block.h).  Records are
// written in (tet, face, tile) order and the stable sort keeps that order for equal depth keys.  The sort moves
// record indices; the tile renderers read the records through them.
#include "bin_block.h"
#include "sort_plan.h"

namespace dtv {

// One workgroup per kTets tets of the batch's block grid.
template <int kTets>
__global__ __launch_bounds__(kBinBlock) void k_bin(const BatchItem* __restrict__ items, int nitems, BinOut out) {
    __shared__ BinLds<kTets> L;
    const uint32_t part = bin_ticket(L, out.scratch);
    const BatchItem& B = items[item_of_block(items, nitems, part / (kBinUnit / kTets))];
    const ViewUniforms& U = B.U;
    const int64_t tet = (int64_t)part * kTets - (int64_t)B.block0 * kBinUnit + threadIdx.x;
    ProjectedTet PT;
    PT.culled = true;
    PT.visible = 0;
    if (threadIdx.x < kTets && tet < B.T) project_tet(U, B.cells, B.pos, tet, PT);
    const uint32_t visible = PT.culled ? 0u : PT.visible;
    uint32_t nfaces;
    uint32_t e = block_exclusive_scan<kBinBlock>((uint32_t)__popc(visible), L.tmp, nfaces);
    uint32_t kmin = 0xFFFFFFFFu, kmax = 0u;
    if (visible)
#pragma unroll
        for (int v = 0; v < 4; v++) bin_vertex(U, L, v, PT.ndc[v][0], PT.ndc[v][1]);
#pragma unroll
    for (int f = 0; f < 4; f++) {
        if (!(visible & (1u << f))) continue;
        const uint32_t k = face_key(PT, f);
        if (bin_entry(U, L, e, (uint32_t)f, kFaceTable[f][0], kFaceTable[f][1], kFaceTable[f][2], k, 0u)) {
            kmin = min(kmin, k);
            kmax = max(kmax, k);
        }
        e++;
    }
    bin_stats(out.scratch, part, (uint32_t)__popc(visible), kmin, kmax);
    bin_emit<true>(B, L, nfaces, part, gridDim.x, out);
}

// ranges[t] = the sorted records of tile t; masks (kMasks): their coverage masks in sorted order, from the last uint4
// of each record of rec_len.
template <bool kMasks>
__global__ __launch_bounds__(256) void k_tile_ranges(const SortRoute* __restrict__ route, int64_t n_cap,
                                                     const uint64_t* __restrict__ n_dev, uint2* __restrict__ ranges,
                                                     const uint4* __restrict__ recs, int rec_len) {
    const uint32_t* __restrict__ keys = route->keys;
    const uint32_t* __restrict__ vals = route->vals;
    uint2* __restrict__ masks = route->masks;
    const uint32_t shift = route->tile_shift;
    const int64_t n = run_count(n_cap, n_dev);
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const uint32_t t = tile_of_key(keys[i], shift);
        if (i == 0 || tile_of_key(keys[i - 1], shift) != t) ranges[t].x = (uint32_t)i;
        if (i == n - 1 || tile_of_key(keys[i + 1], shift) != t) ranges[t].y = (uint32_t)(i + 1);
        if constexpr (kMasks) {
            const uint4 r = recs[rec_len * ((int64_t)vals[i] + 1) - 1];
            masks[i] = make_uint2(r.y, r.z);
        }
    }
}

// Tile launch order, heaviest first.  A tile's rendering time grows with its records and fragments, and tiles are
// handed to the CUs in workgroup order: in row-major order the heavy tiles of the image centre start mid-launch
// and the last of them finish long after the rest of the GPU has gone idle.  Started first, the light tiles fill
// in behind them.  Costs are ranked coarsely (8 buckets per octave, 256 buckets for 32 bits).
__device__ __forceinline__ uint32_t cost_bucket(uint32_t c) {
    const uint32_t v = c < 0xFFFFFFFFu ? c + 1u : c;  // >= 1
    const int e = 31 - __clz((int)v);
    const uint32_t m = e >= 3 ? (v >> (e - 3)) & 7u : (v << (3 - e)) & 7u;
    return 8u * (uint32_t)e + m;
}

// Tiles per thread per step: their costs are loaded together, so the loads overlap (one step per pass up to
// 16K tiles, a 1024x1024 view).
constexpr int kOrderPer = 16;

// Adds one to counter[b] for every live lane and returns the count before it.  Tiles without cost share one bucket
// and are many, so their lanes are added together (LDS atomics on one address serialise); the others spread over
// the buckets.  Every lane of the wave must take part.
__device__ __forceinline__ uint32_t bucket_add(uint32_t* counter, bool live, uint32_t b) {
    const bool empty = live && b == 0u;
    const uint64_t m = ballot(empty);
    const uint32_t below = (uint32_t)popc64(m & lanemask_lt());
    uint32_t at = 0u;
    if (live && (!empty || below == 0u)) at = atomicAdd(&counter[b], empty ? (uint32_t)popc64(m) : 1u);
    const int leader = m != 0ull ? __builtin_ctzll(m) : 0;
    const uint32_t at0 = (uint32_t)__shfl((int)at, leader, 64);
    return empty ? at0 + below : at;
}

__device__ __forceinline__ void load_buckets(const uint2* __restrict__ ranges, const uint32_t* __restrict__ cost,
                                             uint32_t i0, uint32_t n, uint32_t b[kOrderPer]) {
    uint32_t c[kOrderPer];
#pragma unroll
    for (int q = 0; q < kOrderPer; q++) {
        const uint32_t i = i0 + 1024u * q + threadIdx.x;
        c[q] = 0u;
        if (i < n) c[q] = cost != nullptr ? cost[i] : ranges[i].y - ranges[i].x;
    }
#pragma unroll
    for (int q = 0; q < kOrderPer; q++) b[q] = cost_bucket(c[q]);
}

__global__ __launch_bounds__(1024) void k_tile_order(const uint2* __restrict__ ranges,
                                                     const uint32_t* __restrict__ cost, uint32_t n,
                                                     uint32_t* __restrict__ order) {
    __shared__ uint32_t count[256], start[256];
    const uint32_t t = threadIdx.x;
    if (t < 256) count[t] = 0u;
    __syncthreads();
    // trip counts are uniform over the workgroup, so every lane of a wave reaches the ballots
    for (uint32_t i0 = 0; i0 < n; i0 += 1024u * kOrderPer) {
        uint32_t b[kOrderPer];
        load_buckets(ranges, cost, i0, n, b);
#pragma unroll
        for (int q = 0; q < kOrderPer; q++) {
            if (i0 + 1024u * q >= n) break;  // uniform
            (void)bucket_add(count, i0 + 1024u * q + t < n, b[q]);
        }
    }
    __syncthreads();
    if (t < 64) {
        // start[b] = tiles in the buckets above b; lane l takes buckets 255 - 4l down to 252 - 4l
        uint32_t c[4], sum = 0u;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            c[k] = count[255 - 4 * t - k];
            sum += c[k];
        }
        uint32_t run = wave_inclusive_scan(sum) - sum;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            start[255 - 4 * t - k] = run;
            run += c[k];
        }
    }
    __syncthreads();
    for (uint32_t i0 = 0; i0 < n; i0 += 1024u * kOrderPer) {
        uint32_t b[kOrderPer];
        load_buckets(ranges, cost, i0, n, b);
#pragma unroll
        for (int q = 0; q < kOrderPer; q++) {
            if (i0 + 1024u * q >= n) break;  // uniform
            const uint32_t i = i0 + 1024u * q + t;
            const uint32_t at = bucket_add(start, i < n, b[q]);
            if (i < n) order[at] = i;
        }
    }
}

// cost[g] = records of the binning tile that holds 8x8 sub-tile g (the forward's launch order for binning tiles
// larger than 8x8, whose records every sub-tile of the tile walks).
__global__ __launch_bounds__(256) void k_subtile_cost(const BatchItem* __restrict__ items, int nitems, int64_t nsub,
                                                       const uint2* __restrict__ ranges, uint32_t* __restrict__ cost) {
    const int64_t g = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (g >= nsub) return;
    const BatchItem& B = items[item_of_sub(items, nitems, (uint32_t)g)];
    const ViewUniforms& U = B.U;
    const int sub = (int)((uint32_t)g - B.sub0);
    const int k = U.tile_shift - 3;
    const uint32_t t = B.tile0 + (uint32_t)(((sub / U.sub_x) >> k) * U.tiles_x + ((sub % U.sub_x) >> k));
    const uint2 r = ranges[t];
    cost[g] = r.y - r.x;
}

// tile_frags[g] = fragments composited in 8x8 sub-tile g, from the pixels' counts.  One wave per sub-tile.
__global__ __launch_bounds__(64) void k_tile_frags(const BatchItem* __restrict__ items, int nitems,
                                                   const uint32_t* __restrict__ frag_count,
                                                   uint32_t* __restrict__ tile_frags) {
    const BatchItem& B = items[item_of_sub(items, nitems, blockIdx.x)];
    const ViewUniforms& U = B.U;
    const int sub = (int)(blockIdx.x - B.sub0), lane = threadIdx.x;
    const int x = 8 * (sub % U.sub_x) + (lane & 7), y = 8 * (sub / U.sub_x) + (lane >> 3);
    const uint32_t n = x < U.width && y < U.height ? frag_count[B.pixel0 + (int64_t)y * U.width + x] : 0u;
    const uint32_t all = wave_sum_u32(n);
    if (lane == 0) tile_frags[blockIdx.x] = all;
}

void launch_tile_frags(const BatchItem* items, int nitems, int64_t nsub, PixelState ps, hipStream_t s) {
    if (nsub <= 0) return;
    hipLaunchKernelGGL(k_tile_frags, dim3((unsigned)nsub), dim3(64), 0, s, items, nitems, ps.frag_count, ps.tile_frags);
}

void launch_subtile_cost(const BatchItem* items, int nitems, int64_t nsub, const uint2* ranges, uint32_t* cost,
                         hipStream_t s) {
    if (nsub <= 0) return;
    hipLaunchKernelGGL(k_subtile_cost, dim3((unsigned)((nsub + 255) / 256)), dim3(256), 0, s, items, nitems, nsub,
                       ranges, cost);
}

int64_t bin_blocks(int64_t T) { return T > 0 ? (T + kBinUnit - 1) / kBinUnit : 0; }
int64_t bin_status_words(int64_t nblocks) { return 4 * nblocks + 1; }

// A workgroup of 64 tets keeps all threads busy where a tet has many candidate tiles, and makes more workgroups of a
// small mesh; of fine meshes it makes too many (a ticket costs about 14 ns).  Measured, 64 / 256 tets, us: 24,576
// tets at 256^2 43 / 62, ball of 132K tets at 768^2 131 / 201, 196K tets at 1024^2 162 / 242, 1.57M at 2048^2 829 /
// 1143; 196K at 507x389 103 / 76, 400K-tet ball at 512^2 159 / 151, 1.57M at 1024^2 515 / 402, 16 such views at
// 512^2 5429 / 3033.
bool bin_small(int64_t tets, int64_t pixels) { return tets <= 65536 || 4 * pixels >= 5 * tets; }

void launch_bin(const BatchItem* items, int nitems, int64_t nblocks, bool small, const BinOut& out, hipStream_t s) {
    if (nblocks <= 0) return;
    if (small)
        hipLaunchKernelGGL(k_bin<64>, dim3((unsigned)(4 * nblocks)), dim3(kBinBlock), 0, s, items, nitems, out);
    else
        hipLaunchKernelGGL(k_bin<256>, dim3((unsigned)nblocks), dim3(kBinBlock), 0, s, items, nitems, out);
}

void launch_tile_ranges(const SortRoute* route, int64_t n, const uint64_t* n_dev, uint2* ranges, const uint4* recs,
                        int rec_len, hipStream_t s) {
    if (n <= 0) return;
    int64_t blocks = (n + 255) / 256;
    if (blocks > 8192) blocks = 8192;
    if (recs != nullptr)
        hipLaunchKernelGGL(k_tile_ranges<true>, dim3((unsigned)blocks), dim3(256), 0, s, route, n, n_dev, ranges, recs,
                           rec_len);
    else
        hipLaunchKernelGGL(k_tile_ranges<false>, dim3((unsigned)blocks), dim3(256), 0, s, route, n, n_dev, ranges,
                           recs, rec_len);
}

void launch_tile_order(const uint2* ranges, const uint32_t* cost, int64_t num_tiles, uint32_t* order,
                       hipStream_t s) {
    if (num_tiles <= 0) return;
    hipLaunchKernelGGL(k_tile_order, dim3(1), dim3(1024), 0, s, ranges, cost, (uint32_t)num_tiles, order);
}

}  // namespace dtv
