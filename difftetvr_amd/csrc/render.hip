// Tile renderer and its adjoint on gfx950.
//
// One wave64 per 8x8 screen tile, or, for viewports of few tiles, several that take 4x4 or 2x2 pixels each.  The
// tile's sorted (tile, face) records are consumed in batches of 32: each lane stages one record in LDS (tet vertices,
// colours, face planes); the records' coverage masks, exact from binning, give every lane (pixel) a 32-bit mask of the
// records that cover it.  The masks become a dense list of (pixel, record) fragments in LDS, and the expensive
// per-fragment work (ray-tet intersection, barycentric colours, four sub-segment integrals; in the adjoint also
// their derivatives) runs over that list with every lane busy, in rounds.  Only the cheap per-pixel
// compositing (or, in the adjoint, the inversion of the 'over' operator) walks each pixel's fragments in order.
//
// Reference maths (Data/Shaders/...):
//   ray through pixel centre           Intersect/IntersectRasterization.glsl:141-144
//   ray-tet entry/exit                 Intersect/RayIntersectionTests.glsl:78-106
//   barycentric colours                Common/BarycentricInterpolation.glsl:29-38
//   4 sub-segments, accumulateLinearConst  IntersectRasterization.glsl:228-241, Common/ForwardCommon.glsl:42-49
//   early ray termination              PPLL/Forward.glsl:168-173
// The adjoint re-traverses each pixel back to front from the stored final colour, inverting the 'over'
// operator per tet (the inversion of AdjointIntersectRasterization.glsl:213-228) and resetting to stored
// checkpoints (every K fragments, to bound inversion drift, and before a fragment that takes the transmittance below
// kTinyT, whose input could not be recovered).  Gradients of the 4 tet vertices are reduced per record, then
// per vertex of a batch, in LDS before one global atomic per value.
#include <map>
#include <mutex>

#include "render_common.h"
#include "vertex_table.h"

namespace dtv {

constexpr int kRoundDefault = 128;          // fragments shaded per round of the forward (segments per pass)
constexpr int kRoundAdj = 64;               // fragments per round in the adjoint: one per lane
constexpr float kMissMarker = -1.0f;        // transmittance slot of a fragment whose ray missed the tet
constexpr float kTinyT = 0x1p-100f;         // transmittance below which a fragment's input is not recovered

// The forward's fragment list and round values (kRound fragments shaded per round).  The forward waits on latency (the
// long dependent chain of one fragment's evaluation) more than on issue slots: with the records, rounds of 128 and less
// take 10 KB of LDS and 128 registers, so that four waves fit in each SIMD (a CU has 160 KB).  For that a batch of more
// than kFwdFrags fragments is listed and shaded in several goes, ray directions move between lanes by permute, and the
// vertex indices stay out of the staged records.  Against three waves (13.4 KB, 140 registers): a render of 5.3M tets
// at 1920 x 1080 4.80 -> 4.24 ms, a burst of 24 server requests 8.82 -> 7.60 ms, the step of 1.57M tets at 1024 x 1024
// 6.91 -> 6.62 ms.
constexpr int kFwdFrags = 1024;
template <int kRound>
struct FragListLds {
    uint16_t entry[kFwdFrags];  // (pixel lane << 5) | record index
    float4 val[kRound];         // fragment colour F
};

// The adjoint's: with the records, 13,312 B per wave.  The LDS is handed out in granules of 1,280 B, so a CU's 160 KB
// hold 11 such workgroups (12 up to 12,800 B each), where the registers would allow three waves per SIMD.  A batch
// whose fragments exceed kAdjFrags is processed in two parts of 16 records; the per-fragment gradient rows are reduced
// half a round (32 fragments) at a time; ray directions stay in registers and move between lanes by permute.  The
// flush's vertex table spans entry and w, which are free by then.
constexpr int kAdjFrags = 1024;
struct AdjFragLds {
    uint16_t entry[kAdjFrags];  // (pixel lane << 5) | record index, one part of a batch
    float w[32][29];            // gradient rows of half a round, one per lane (29: conflict-free column access)
    float4 val[kRoundAdj];      // F, then dL/dF (.w: d/d(alpha), alpha = 1 - F.w); w = kMissMarker on a miss
};

// Ray direction of pixel lane pl from the lanes' own (register) directions; every lane must take part.
__device__ __forceinline__ float3_ lane_ray(float3_ mine, int pl) {
    return f3(__shfl(mine.x, pl, 64), __shfl(mine.y, pl, 64), __shfl(mine.z, pl, 64));
}

// kCell: renders the items with per-cell colours (BatchItem::cell_col), else those with per-vertex colours; a
// batch that holds both is rendered by one launch of each, every tile by the one matching its item.
// kRound: fragments shaded per round (64, 128 or 256: segments per pass).  kSub: binning tiles larger than 8x8
// (the workgroup's 8x8 sub-tile tests its own coverage).  kEdge < 8: this wave renders part `part` of the tile
// (PartOfTile).
template <bool kCell, int kRound, bool kSub, int kEdge = kTileEdge>
__device__ __forceinline__ void forward_tile(const BatchItem* __restrict__ items, int nitems,
                                             RecordStream stream, const uint2* __restrict__ ranges,
                                             const PixelState& ps_all, uint32_t gsub, RecordLds& L,
                                             FragListLds<kRound>& F, uint32_t part = 0u) {
    constexpr bool kPart = kEdge < kTileEdge;
    static_assert(!(kPart && kSub), "parts of 8x8 binning tiles only");
    const BatchItem& B = items[item_of_sub(items, nitems, gsub)];
    if ((B.cell_col != nullptr) != kCell) return;
    const ViewUniforms& U = B.U;
    const float* __restrict__ pos = B.pos;
    const float* __restrict__ col = kCell ? B.cell_col : B.col;
    float4* __restrict__ out_image = reinterpret_cast<float4*>(B.image);
    const PixelState ps = item_pixel_state(ps_all, B);
    const SubTile st = sub_tile(B, gsub);
    const uint32_t gtile = st.gtile;
    const int lane = threadIdx.x;
    const uint64_t lt = lanemask_lt();
    const PartOfTile<kEdge> pt(part);
    const int lx = lane % kEdge, ly = lane / kEdge;
    const int x = st.x0 + pt.x0 + lx, y = st.y0 + pt.y0 + ly;
    // binning tiles larger than 8x8: coverage is tested here, from face triangles stashed in the fragment
    // list's space (free while a batch is staged)
    int32_t* stash = kSub ? reinterpret_cast<int32_t*>(F.entry) : nullptr;
    const bool valid = lane < pt.kPixels && x < U.width && y < U.height;
    if (kPart && ballot(valid) == 0ull) return;
    const float3_ ro = f3(U.camPos[0], U.camPos[1], U.camPos[2]);
    const float3_ my_rd = ray_direction(U, x, y);
    const float my_scale = seg_scale(U, my_rd);
    const float att = U.attenuation;
    const uint2 rg = ranges[gtile];
    const int P = U.width * U.height;
    const int pix = valid ? pixel_index(U, x, y) : 0;

    float4 C = make_float4(0.f, 0.f, 0.f, 1.0f);  // premultiplied RGB, transmittance
    uint32_t n = 0, last = rg.x, nck = 0, nlast = 0;
    bool done = !valid;
    // Three-stage prefetch: while a batch is shaded, the next batch's vertex data, the record words of the batch
    // after it and the record indices of the one after that (of a part: its candidates' masks) are in flight.
    RecordIn cur, nxt;
    RecordData cd;
    const uint4* __restrict__ recs = stream.recs;
    const uint32_t* __restrict__ rec_of = stream.route->vals;
    PartFeed<kEdge, false> feed{recs, rec_of, stream.route->masks, rg.x, rg.y, pt.origin, {}};
    uint32_t ahead = 0u;  // this lane's record of the batch after nxt's
    // a part's batch: the stream indices of its records (the entries of a part fill at most half the list)
    static_assert(!kPart || PartOfTile<kEdge>::kPixels * kBatch <= kFwdFrags / 2, "no room for a part's indices");
    uint32_t* const part_idx = reinterpret_cast<uint32_t*>(F.entry + kFwdFrags / 2);
    uint32_t* const pend = part_idx + kBatch;
    uint32_t cur_idx = 0u, nxt_idx = 0u;
    int ncur = 0, nnxt = 0;
    if constexpr (kPart) {
        feed.load(lane);
        ncur = feed.next(pend, lane, cur, cur_idx);
        feed.load(lane);
        if (lane < ncur) fetch_record_data<kCell>(pos, col, cur, cd);
        nnxt = feed.next(pend, lane, nxt, nxt_idx);
        feed.load(lane);
    } else {
        if (lane < kBatch && rg.x + kBatch + lane < rg.y) nxt = load_record(recs, rec_of[rg.x + kBatch + lane]);
        if (lane < kBatch && rg.x + lane < rg.y) {
            cur = load_record(recs, rec_of[rg.x + lane]);
            fetch_record_data<kCell>(pos, col, cur, cd);
        }
        if (lane < kBatch && rg.x + 2 * kBatch + lane < rg.y) ahead = rec_of[rg.x + 2 * kBatch + lane];
    }
    for (uint32_t base = rg.x; kPart ? ncur > 0 : base < rg.y; base += kBatch) {
        const int cnt = kPart ? ncur : (int)min((uint32_t)kBatch, rg.y - base);
        if (lane < cnt) store_record<kSub>(U, cur, cd, L, lane, stash);
        uint32_t mask;
        if constexpr (kPart) {
            if (lane < cnt) part_idx[lane] = cur_idx;
            mask = pt.coverage(cur.rec, cnt, lane);
            if (done) mask = 0u;
            cur = nxt;
            cur_idx = nxt_idx;
            ncur = nnxt;
            if (lane < ncur) fetch_record_data<kCell>(pos, col, cur, cd);
            nnxt = feed.next(pend, lane, nxt, nxt_idx);
            feed.load(lane);
            __syncthreads();
        } else {
            if (lane < kBatch && base + kBatch + lane < rg.y) {
                cur = nxt;
                fetch_record_data<kCell>(pos, col, cur, cd);
            }
            if (lane < kBatch && base + 2 * kBatch + lane < rg.y) nxt = load_record(recs, ahead);
            if (lane < kBatch && base + 3 * kBatch + lane < rg.y) ahead = rec_of[base + 3 * kBatch + lane];
            __syncthreads();
            if constexpr (kSub) {
                subtile_masks(L, stash, cnt, x, y, valid, lane);
                __syncthreads();
            }
            mask = done ? 0u : lane_coverage(L, cnt, lane);
        }
        // the records' coverage masks are consumed: their slots hold the list's rank masks
        uint64_t* rank_mask = reinterpret_cast<uint64_t*>(&L.mask[0][0]);
        do {  // one list, or several where the batch has more fragments than it holds
            const uint32_t before = (uint32_t)__popc(mask);
            const uint32_t total = build_fragment_list<kFwdFrags>(F.entry, rank_mask, mask, lane);
            const uint32_t nmine = before - (uint32_t)__popc(mask);
            RankCursor cur_e;
            __syncthreads();
            for (uint32_t r0 = 0; r0 < total; r0 += kRound) {
                for (uint32_t i0 = 0; i0 < (uint32_t)kRound && r0 + i0 < total; i0 += 64) {
                    // lanes behind the list's end evaluate the last fragment again
                    const uint32_t i = i0 + lane;
                    const uint32_t ent = F.entry[min(r0 + i, total - 1u)];
                    const int pl = ent >> 5, j = ent & 31;
                    const float3_ rdp = lane_ray(my_rd, pl);
                    const float tscale = U.linear_depth ? __shfl(my_scale, pl, 64) : 1.0f;
                    FragEval E;
                    eval_fragment<kCell, false>(L, j, ro, rdp, att, tscale, E);
                    F.val[i] = E.hit ? E.F : make_float4(0.f, 0.f, 0.f, kMissMarker);
                }
                __syncthreads();
                uint32_t e;
                while (!done && cur_e.next(rank_mask, nmine, lt, r0 + kRound, e)) {
                    if (U.use_ert && (1.0f - C.w) > U.ert_alpha) {
                        done = true;
                        break;
                    }
                    const float4 f = F.val[e - r0];
                    // C.w is the transmittance T, the product of the fragments' transmittances (relative precision at
                    // any depth), so the adjoint recovers each fragment's input as T_out / T_f.  Only an underflow
                    // (T_out below kTinyT) cannot be inverted: a checkpoint goes before the fragment that causes it.
                    // The state before the first fragment (T = 1) needs no slot.  A missed fragment's value is
                    // (0, 0, 0, kMissMarker): with transmittance 1 it leaves the state as it is, without a branch.
                    const float Tout = C.w * (f.w != kMissMarker ? f.w : 1.0f);
                    if (C.w >= kTinyT && Tout < kTinyT && nlast != n && (int)nck < U.max_ckpt) {
                        ps.ckpt_t[(int64_t)nck * P + pix] = C.w;
                        ps.ckpt_n[(int64_t)nck * P + pix] = n;
                        nck++;
                        nlast = n;
                    }
                    {
#pragma clang fp contract(fast)
                        C.x = C.x + C.w * f.x;
                        C.y = C.y + C.w * f.y;
                        C.z = C.z + C.w * f.z;
                    }
                    C.w = Tout;
                    n++;
                    last = (kPart ? part_idx[F.entry[e] & 31] : base + (F.entry[e] & 31)) + 1;
                    // periodic checkpoints bound the rounding the adjoint's chain of divisions accumulates; the last
                    // slot is kept for the underflow rule above
                    if ((int)(n - nlast) >= U.ckpt_interval && C.w >= kTinyT && (int)nck < U.max_ckpt - 1) {
                        ps.ckpt_t[(int64_t)nck * P + pix] = C.w;
                        ps.ckpt_n[(int64_t)nck * P + pix] = n;
                        nck++;
                        nlast = n;
                    }
                }
                __syncthreads();
            }
        } while (ballot(mask != 0u) != 0ull);
        if (ballot(!done) == 0ull) break;
    }
    if (valid) {
        const float T = C.w;
        out_image[pix] = make_float4(C.x + T * U.clear[0], C.y + T * U.clear[1], C.z + T * U.clear[2],
                                     (1.0f - T) + T * U.clear[3]);
        ps.ray_color[pix] = C;
        ps.frag_count[pix] = n;
        ps.last_rec[pix] = last;
        ps.num_ckpt[pix] = nck;
    }
    // the tile's composited fragments: the adjoint's launch order ranks tiles by them (parts are not ranked)
    if constexpr (!kPart) {
        const uint32_t tile_total = wave_inclusive_scan(n);
        if (lane == 63) ps.tile_frags[gsub] = tile_total;
    }
}

// Next entry of the launch order for a persistent workgroup: one claim per tile from the launch's queue
// counter (zeroed before the launch), uniform across the wave.  Every tile is claimed, none assigned by block
// index: a workgroup the GPU cannot hold at first (the occupancy estimate is an upper bound) starts only when
// another exits, and must not be holding a tile meanwhile.
__device__ __forceinline__ uint32_t claim_tile(uint32_t* __restrict__ queue) {
    uint32_t t = 0;
    if (threadIdx.x == 0) t = atomicAdd(queue, 1u);
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)__shfl((int)t, 0, 64));
}

// kQueue = false: one workgroup per tile of the launch order.  kQueue = true: as many workgroups as the GPU
// holds at once, each claiming the next tile of the launch order from `queue` until all ntiles are taken.
template <bool kCell, int kRound, bool kSub, bool kQueue>
__global__ __launch_bounds__(64, kRound > 128 ? 3 : 4) void k_render_forward(const BatchItem* __restrict__ items, int nitems,
                                                        const uint32_t* __restrict__ order,
                                                        RecordStream stream,
                                                        const uint2* __restrict__ ranges, PixelState ps_all,
                                                        uint32_t* __restrict__ queue, uint32_t ntiles) {
    __shared__ RecordLds L;
    __shared__ FragListLds<kRound> F;
    if constexpr (!kQueue) {
        forward_tile<kCell, kRound, kSub>(items, nitems, stream, ranges, ps_all, global_tile_of_block(order), L, F);
    } else {
        for (uint32_t t = claim_tile(queue); t < ntiles; t = claim_tile(queue)) {
            forward_tile<kCell, kRound, kSub>(items, nitems, stream, ranges, ps_all,
                                              order != nullptr ? order[t] : t, L, F);
            __syncthreads();
        }
    }
}

// (8 / kEdge)^2 workgroups per tile, one per part, in image order.
template <bool kCell, int kEdge>
__global__ __launch_bounds__(64, 4) void k_render_forward_parts(const BatchItem* __restrict__ items, int nitems,
                                                              RecordStream stream,
                                                              const uint2* __restrict__ ranges, PixelState ps_all) {
    __shared__ RecordLds L;
    __shared__ FragListLds<kRoundDefault> F;
    constexpr uint32_t kParts = PartOfTile<kEdge>::kParts;
    forward_tile<kCell, kRoundDefault, false, kEdge>(items, nitems, stream, ranges, ps_all, blockIdx.x / kParts, L, F,
                                                     blockIdx.x % kParts);
}

// What bounds it: vector instructions and the LDS together (1,572,864 tets at 1024 x 1024, 76.1 M listed fragments in
// 1.32 M rounds: 1.82e9 instructions, about 1,380 a round of up to 64 fragments, 82 % of one per SIMD and four cycles;
// the LDS 68 % busy); memory traffic matters little, and three waves per SIMD are all that the registers of a
// fragment's gradients allow (10.7 of the 11 workgroups a CU that fit are resident; four waves, with rows of a quarter
// round and 77 spills, made steps 2 to 10 % slower).  So the phases are written for few instructions: A and C without
// branches, the checkpoint test of B as one comparison, the owners' row masks for both halves of a round from one set
// of ballots, the flush as LDS additions of doubles (2.19e9 -> 2.02e9 instructions in all, the whole step 7.80 -> 7.62
// ms, and 1.02 to 1.04 times faster from 24K tets on), and the sub-segments' adjoint as running sums shared with the
// composite (frag_backward_exact: a fragment's backward 537 -> 432 instructions; the step 7.04 -> 6.90 ms).
//
// kRef = false: exact derivative of the forward.  kRef = true: the reference's adjoint as written
// (AdjointIntersectRasterization.glsl:111-362): per pixel from the blended output image, back to front, the
// 'over' operator is inverted per sub-segment 3, 2, 1 (sub-segment 0 is skipped) with no checkpoints, and
// each fragment's parameter gradients follow frag_backward_reference.
// kCell: the items with per-cell colours (exact adjoint only), kSub: binning tiles larger than 8x8, kEdge < 8: a
// part of the tile, as k_render_forward.
template <bool kRef, bool kCell, bool kSub, int kEdge = kTileEdge>
__device__ __forceinline__ void adjoint_tile(const BatchItem* __restrict__ items,
                                             const AdjointTarget* __restrict__ targets, int nitems,
                                             RecordStream stream, const uint2* __restrict__ ranges,
                                             const PixelState& ps_all, int use_abs, uint32_t gsub, RecordVidLds& L,
                                             AdjFragLds& A, float4 (&s_seg)[kRef ? 3 : 1][kRoundAdj],
                                             uint32_t part = 0u) {
    constexpr bool kPart = kEdge < kTileEdge;
    static_assert(!(kPart && kSub), "parts of 8x8 binning tiles only");
    const int item = item_of_sub(items, nitems, gsub);
    const BatchItem& B = items[item];
    if ((B.cell_col != nullptr) != kCell) return;
    const ViewUniforms& U = B.U;
    const float* __restrict__ pos = B.pos;
    const float* __restrict__ col = kCell ? B.cell_col : B.col;
    const float4* __restrict__ dimage = reinterpret_cast<const float4*>(targets[item].dimage);
    if (dimage == nullptr) return;  // item not differentiated
    // positions and vertex colours accumulate in the item's interleaved rows (8 floats per vertex: xyz, rgba)
    float* __restrict__ vacc = targets[item].acc;
    float* __restrict__ grad_col = targets[item].grad_col;  // per-cell colours: straight to the tet
    const PixelState ps = item_pixel_state(ps_all, B);
    const SubTile st = sub_tile(B, gsub);
    const uint32_t gtile = st.gtile;
    const int lane = threadIdx.x;
    const PartOfTile<kEdge> pt(part);
    const int lx = lane % kEdge, ly = lane / kEdge;
    const int x = st.x0 + pt.x0 + lx, y = st.y0 + pt.y0 + ly;
    const bool valid = lane < pt.kPixels && x < U.width && y < U.height;
    int32_t* stash = kSub ? reinterpret_cast<int32_t*>(A.entry) : nullptr;
    const float3_ ro = f3(U.camPos[0], U.camPos[1], U.camPos[2]);
    const float3_ my_rd = ray_direction(U, x, y);
    const float my_scale = seg_scale(U, my_rd);
    const float att = U.attenuation;
    const uint2 rg = ranges[gtile];
    const int P = U.width * U.height;
    const int pix = valid ? pixel_index(U, x, y) : 0;

    uint32_t natom = 0;  // gradient atomics this lane issued (counted when ps.counters is set)
    // exact mode: C.w = the transmittance behind the fragment being undone (only it is needed); reference mode:
    // the blended premultiplied RGBA the reference inverts
    float4 C = make_float4(0.f, 0.f, 0.f, 1.0f);
    float dC[4] = {0.f, 0.f, 0.f, 0.f};
    uint32_t n = 0, last = 0;
    CheckpointCursor ck;
    if (valid) {
        C = ps.ray_color[pix];
        n = ps.frag_count[pix];
        last = ps.last_rec[pix];
        if constexpr (!kRef) ck.start((int)ps.num_ckpt[pix], n, C.w, P, ps, pix);
        const float4 di = dimage[pix];
        dC[0] = di.x;
        dC[1] = di.y;
        dC[2] = di.z;
        if constexpr (kRef) {
            // the reference starts from the blended output image and the raw image adjoint
            const float T = C.w;
            C = make_float4(C.x + T * U.clear[0], C.y + T * U.clear[1], C.z + T * U.clear[2],
                            (1.0f - T) + T * U.clear[3]);
            dC[3] = di.w;
        } else {
            dC[3] = di.w * (1.0f - U.clear[3]) - (di.x * U.clear[0] + di.y * U.clear[1] + di.z * U.clear[2]);
        }
    }
    bool done = !valid || n == 0;
    if (ballot(!done) == 0ull) return;
    // Batches run back to front, from the last record that any of the wave's pixels composited (early ray
    // termination leaves the records behind it out).  The next batch's record words are loaded when the current
    // batch starts and its vertex data just before the current batch's gradient atomics, so that staging it never
    // waits on memory (record indices one batch further ahead).
    const uint32_t behind = (uint32_t)__builtin_amdgcn_readfirstlane((int)wave_max_u32(valid ? last : 0u));
    const int nbatch = (int)((behind - rg.x + kBatch - 1) / kBatch);
    RecordIn nxt;
    RecordData nd;
    const uint4* __restrict__ recs = stream.recs;
    const uint32_t* __restrict__ rec_of = stream.route->vals;
    PartFeed<kEdge, true> feed{recs, rec_of, stream.route->masks, rg.x, behind, pt.origin, {}};
    uint32_t ahead = 0u;  // this lane's record of the next batch
    static_assert(!kPart || PartOfTile<kEdge>::kPixels * kBatch <= kAdjFrags / 2, "no room for a part's indices");
    uint32_t* const part_idx = reinterpret_cast<uint32_t*>(A.entry + kAdjFrags / 2);  // as in the forward
    uint32_t* const pend = part_idx + kBatch;
    uint32_t nxt_idx = 0u;
    int nnxt = 0;
    if constexpr (kPart) {
        feed.load(lane);
        nnxt = feed.next(pend, lane, nxt, nxt_idx);
        if (lane < nnxt) fetch_record_data<kCell>(pos, col, nxt, nd);
    } else {
        const uint32_t b0 = rg.x + (uint32_t)(nbatch - 1) * kBatch;
        if (lane < kBatch && b0 + lane < rg.y) {
            nxt = load_record(recs, rec_of[b0 + lane]);
            fetch_record_data<kCell>(pos, col, nxt, nd);
        }
        if (nbatch > 1 && lane < kBatch) ahead = rec_of[b0 - kBatch + lane];
    }
    for (int bi = nbatch - 1; kPart ? nnxt > 0 : bi >= 0; bi--) {
        const uint32_t base = kPart ? 0u : rg.x + (uint32_t)bi * kBatch;
        const int cnt = kPart ? nnxt : (int)min((uint32_t)kBatch, rg.y - base);
        if (lane < cnt) store_record<kSub>(U, nxt, nd, L, lane, stash);
        uint32_t cover = 0u;
        if constexpr (kPart) {
            if (lane < cnt) part_idx[lane] = nxt_idx;
            cover = pt.coverage(nxt.rec, cnt, lane);
            feed.load(lane);
            nnxt = feed.next(pend, lane, nxt, nxt_idx);
        } else if (bi > 0 && lane < kBatch) {
            nxt = load_record(recs, ahead);
            if (bi > 1) ahead = rec_of[base - 2 * kBatch + lane];
        }
        const bool more = kPart ? nnxt > 0 : bi > 0;
        // lanes j and j + 32 own record j's 28 values (first / second half of 14) for this batch
        float acc[14];
#pragma unroll
        for (int q = 0; q < 14; q++) acc[q] = 0.f;
        __syncthreads();
        if constexpr (kSub) {
            subtile_masks(L, stash, cnt, x, y, valid, lane);
            __syncthreads();
        }
        // records at or after `last` were not composited in the forward (early ray termination)
        uint32_t mask_all;
        if constexpr (kPart) {  // slots back to front
            uint32_t dead = 0u;
            while (!done && dead < (uint32_t)cnt && part_idx[dead] >= last) dead++;
            mask_all = done || dead >= 32u ? 0u : cover & (0xFFFFFFFFu << dead);
        } else {
            const uint32_t nlive = last > base ? min((uint32_t)cnt, last - base) : 0u;
            const uint32_t live = nlive >= 32u ? 0xFFFFFFFFu : ((1u << nlive) - 1u);
            mask_all = done ? 0u : (lane_coverage(L, cnt, lane) & live);
        }
        // parts (back to front): all 32 records, or records 16-31 then 0-15 when the list exceeds kAdjFrags
        int nparts = 1;
        if constexpr (!kPart) {
            const uint32_t inc = wave_inclusive_scan((uint32_t)__popc(mask_all));
            if ((uint32_t)__builtin_amdgcn_readlane((int)inc, 63) > (uint32_t)kAdjFrags) nparts = 2;
        }
        for (int part = 0; part < nparts; part++) {
        const uint32_t pmask = nparts == 1 ? 0xFFFFFFFFu : (part == 0 ? 0xFFFF0000u : 0x0000FFFFu);
        const uint32_t mask = done ? 0u : (mask_all & pmask);
        uint32_t total;
        const uint32_t off = build_fragment_list_by_pixel(A.entry, mask, !kPart, lane, total);
        const uint32_t mine_end = off + (uint32_t)__popc(mask);
        __syncthreads();
        for (uint32_t r0 = 0; r0 < total; r0 += kRoundAdj) {
            // A: fragment colours (one fragment per lane; E stays in registers for phase C).  The exact adjoint's
            // phases A and C run without branches: a lane behind the list's end evaluates the last fragment again
            // and drops the result, so no register has to be cleared for it.
            FragEval E;
            E.hit = false;
            {
                const uint32_t e = r0 + lane;
                const uint32_t ent = A.entry[min(e, total - 1u)];
                const int pl = ent >> 5, j = ent & 31;
                const float3_ rdp = lane_ray(my_rd, pl);
                const float tscale = U.linear_depth ? __shfl(my_scale, pl, 64) : 1.0f;
                if (!kRef || e < total) {
                    eval_fragment<kCell, true, kRef>(L, j, ro, rdp, att, tscale, E);
                    A.val[lane] = E.hit ? E.F : make_float4(0.f, 0.f, 0.f, kMissMarker);
                    if constexpr (kRef) {
#pragma unroll
                        for (int s = 1; s < 4; s++) s_seg[s - 1][lane] = E.seg[s];
                    }
                }
            }
            __syncthreads();
            // B: per pixel, back to front: undo the composite, dL/dF of each fragment
            const uint32_t e0 = max(off, r0), e1 = min(mine_end, r0 + kRoundAdj);
            for (uint32_t e = e0; e < e1; e++) {
                if constexpr (kRef) {
                    // reference: invert sub-segments 3..1 of the fragment; dL/d(sub-segment colour) replaces
                    // the sub-segment colour in s_seg (AdjointIntersectRasterization.glsl:204-228)
                    if (A.val[e - r0].w != kMissMarker) {
#pragma unroll
                        for (int s = 3; s > 0; s--) {
                            const float4 acc = s_seg[s - 1][e - r0];
                            const float ain = (acc.w - C.w) / (acc.w - 1.0f);
                            const float4 cin = make_float4(C.x - (1.0f - ain) * acc.x, C.y - (1.0f - ain) * acc.y,
                                                           C.z - (1.0f - ain) * acc.z, ain);
                            s_seg[s - 1][e - r0] = make_float4((1.0f - ain) * dC[0], (1.0f - ain) * dC[1],
                                                               (1.0f - ain) * dC[2], (1.0f - ain) * dC[3]);
                            dC[3] = dC[3] * (1.0f - acc.w) - (dC[0] * acc.x + dC[1] * acc.y + dC[2] * acc.z);
                            C = cin;
                        }
                    }
                    n--;
                    continue;
                }
                const float4 f = A.val[e - r0];
                // the fragment's input transmittance: a checkpoint, 1 before the first fragment, or the output
                // divided by the fragment's transmittance (a corrected quotient: the rounding compounds along the
                // chain back to the next checkpoint).  Below kTinyT the forward's rule leaves no checkpoint only
                // where the input was below kTinyT too: that fragment's contribution (at most kTinyT |dL/dI|) is
                // dropped.  Formed without branches; a missed fragment (f.w = kMissMarker) keeps the state, and
                // its slot's value is not read.
                const bool hit = f.w != kMissMarker;
                float Tin = C.w < kTinyT ? 0.0f : div_nr(C.w, f.w);
                C.w = hit ? Tin : C.w;
                n--;
                if (ck.n1 == n) {
                    Tin = ck.t1;
                    C.w = Tin;
                    ck.advance(P, ps, pix);
                }
                A.val[e - r0] = make_float4(Tin * dC[0], Tin * dC[1], Tin * dC[2], Tin * dC[3]);
                {
#pragma clang fp contract(fast)
                    const float d3 = dC[3] * f.w - (dC[0] * f.x + dC[1] * f.y + dC[2] * f.z);
                    dC[3] = hit ? d3 : dC[3];
                }
            }
            if (n == 0) done = true;
            __syncthreads();
            // C: gradients of the fragments (one per lane).  Each fragment's 28 values are stored into A.w (half
            // a round at a time); the owner lanes of each record then add its rows.
            int key = kBatch;  // record index of this lane's fragment, kBatch = none
            float g[28];  // set where key is
            {
                const uint32_t e = r0 + lane;
                const uint32_t ent = A.entry[min(e, total - 1u)];
                const int pl = ent >> 5, j = ent & 31;
                const float3_ rdp = lane_ray(my_rd, pl);
                const float tscale = U.linear_depth ? __shfl(my_scale, pl, 64) : 1.0f;
                if (!kRef || (e < total && E.hit)) {
                    if constexpr (kRef) {
                        const float4 dacc[3] = {s_seg[0][lane], s_seg[1][lane], s_seg[2][lane]};
                        frag_backward_reference(E, L, j, ro, rdp, att, dacc, use_abs != 0, g);
                    } else if constexpr (kCell) {
                        // positions in the usual slots; the tet's colour gradient in vertex 0's colour slots
                        float lam0[4], lam1[4], dcell[4];
                        float3_ Q0, Q1;
                        frag_backward_cell(E, L, j, rdp, att, tscale, A.val[lane], lam0, lam1, dcell, Q0,
                                           Q1);
                        if (use_abs) {
#pragma unroll
                            for (int ch = 0; ch < 4; ch++) dcell[ch] = fabsf(dcell[ch]);
                            Q0 = f3(fabsf(Q0.x), fabsf(Q0.y), fabsf(Q0.z));
                            Q1 = f3(fabsf(Q1.x), fabsf(Q1.y), fabsf(Q1.z));
                        }
#pragma unroll
                        for (int v = 0; v < 4; v++) {
#pragma clang fp contract(fast)
                            const float l0 = lam0[v], l1 = lam1[v];
                            g[7 * v + 0] = l0 * Q0.x + l1 * Q1.x;
                            g[7 * v + 1] = l0 * Q0.y + l1 * Q1.y;
                            g[7 * v + 2] = l0 * Q0.z + l1 * Q1.z;
                        }
#pragma unroll
                        for (int ch = 0; ch < 4; ch++) {
                            g[3 + ch] = dcell[ch];
                            g[10 + ch] = g[17 + ch] = g[24 + ch] = 0.f;
                        }
                    } else {
                        float lam0[4], lam1[4], dcol0[4], dcol1[4];
                        float3_ Q0, Q1;
                        frag_backward_exact(E, L, j, rdp, att, tscale, A.val[lane], lam0, lam1, dcol0,
                                            dcol1, Q0, Q1);
                        if (use_abs) {
#pragma unroll
                            for (int ch = 0; ch < 4; ch++) {
                                dcol0[ch] = fabsf(dcol0[ch]);
                                dcol1[ch] = fabsf(dcol1[ch]);
                            }
                            Q0 = f3(fabsf(Q0.x), fabsf(Q0.y), fabsf(Q0.z));
                            Q1 = f3(fabsf(Q1.x), fabsf(Q1.y), fabsf(Q1.z));
                        }
#pragma unroll
                        for (int v = 0; v < 4; v++) {
#pragma clang fp contract(fast)
                            const float l0 = lam0[v], l1 = lam1[v];
                            g[7 * v + 0] = l0 * Q0.x + l1 * Q1.x;
                            g[7 * v + 1] = l0 * Q0.y + l1 * Q1.y;
                            g[7 * v + 2] = l0 * Q0.z + l1 * Q1.z;
#pragma unroll
                            for (int ch = 0; ch < 4; ch++) g[7 * v + 3 + ch] = l0 * dcol0[ch] + l1 * dcol1[ch];
                        }
                    }
                    if (kRef || (e < total && E.hit)) key = j;
                }
            }
            // Per half round (the fragments of lanes 0-31, then 32-63): each fragment stores its 28 values in
            // the row of its lane; the owner lanes of record j (j and j + 32) find the record's rows from a mask of
            // the lanes whose key equals j, formed from ballots of the key bits for both halves at once, and add them.
            uint32_t eq[2];
            {
                const uint64_t any = ballot(key < kBatch);
                eq[0] = (uint32_t)any;
                eq[1] = (uint32_t)(any >> 32);
#pragma unroll
                for (int b = 0; b < 5; b++) {
                    const uint64_t ones = ballot((key >> b) & 1);
                    const uint32_t flip = (((uint32_t)lane >> b) & 1u) - 1u;
                    eq[0] &= (uint32_t)ones ^ flip;
                    eq[1] &= (uint32_t)(ones >> 32) ^ flip;
                }
            }
#pragma unroll 1
            for (int h = 0; h < 2; h++) {
                const bool mine = (lane >> 5) == h && key < kBatch;
                if (mine) {
#pragma unroll
                    for (int q = 0; q < 28; q++) A.w[lane & 31][q] = g[q];
                }
                __syncthreads();
                {
                    // two rows per step: 28 independent LDS reads in flight instead of 14
                    const int half = lane >> 5;
                    uint32_t m = h == 0 ? eq[0] : eq[1];
                    while (m) {
                        const int r1 = __ffs(m) - 1;
                        m &= m - 1u;
                        if (m) {
                            const int r2 = __ffs(m) - 1;
                            m &= m - 1u;
                            float a[14], b[14];
#pragma unroll
                            for (int q = 0; q < 14; q++) {
                                a[q] = A.w[r1][half * 14 + q];
                                b[q] = A.w[r2][half * 14 + q];
                            }
#pragma unroll
                            for (int q = 0; q < 14; q++) acc[q] += a[q] + b[q];
                        } else {
#pragma unroll
                            for (int q = 0; q < 14; q++) acc[q] += A.w[r1][half * 14 + q];
                        }
                    }
                }
                __syncthreads();
            }
        }
        }  // parts
        // Flush.  Lanes j and j + 32 hold record j's tet vertices 0, 1 and 2, 3 (7 values each): 128 vertex
        // slots, slot s = v * 32 + j.  Depth-adjacent tets share most vertices (typically 6-7 slots per distinct
        // vertex in a batch), so the slots of one vertex are summed before the global atomics: each slot finds
        // its vertex's entry in an LDS hash table keyed by vertex id (compare-and-swap; the first slot of a
        // vertex creates the entry) and adds its values to the entry's sums.  The sums are doubles: an LDS addition
        // of doubles takes about half a cycle per lane, one of floats about four.  (Rows linked into a list per
        // entry and summed by the entry's creator took 600 vector instructions more per batch, one in eleven of
        // the kernel's.)
        {
            const int j = lane & 31, half = lane >> 5;
            constexpr int kTab = kFlushTab;
            // over entry and w, free after the rounds: sums[kTab][7], keys[kTab]
            double* sums = reinterpret_cast<double*>(&A.entry[0]);
            int32_t* keys = reinterpret_cast<int32_t*>(sums + 7 * kTab);
            static_assert((sizeof(int32_t) + 7 * sizeof(double)) * kTab <= sizeof(A.entry) + sizeof(A.w),
                          "the flush table exceeds the fragment list space");
            static_assert(7 * kTab % 2 == 0 && offsetof(AdjFragLds, w) == sizeof(A.entry), "table layout");
            for (int e = lane; e < 7 * kTab / 2; e += 64)
                reinterpret_cast<double2*>(sums)[e] = make_double2(0.0, 0.0);
            for (int e = lane; e < kTab; e += 64) keys[e] = -1;
            __syncthreads();
            const int s0 = (2 * half) * 32 + j, s1 = s0 + 32;
            const int32_t* vids = &L.vid[0][0];
            const bool slot_live = j < cnt;
            if constexpr (kCell) {
                // the record's tet colour gradient (lane j holds it in vertex 0's colour slots) goes straight
                // to the tet; only positions are merged by vertex below
                if (half == 0 && slot_live) {
                    const int64_t t = L.meta[j] >> 4;
#pragma unroll
                    for (int c = 0; c < 4; c++) {
                        if (acc[3 + c] != 0.f) {
                            atomic_add_f32(&grad_col[4 * t + c], acc[3 + c]);
                            natom++;
                        }
                        acc[3 + c] = 0.f;
                    }
                }
            }
            const int32_t v0 = slot_live ? vids[s0] : 0, v1 = slot_live ? vids[s1] : 0;
            int ent[2] = {-1, -1};
            bool owner[2] = {false, false};
#pragma unroll
            for (int k = 0; k < 2; k++) {
                if (!slot_live) continue;
                const int32_t v = k == 0 ? v0 : v1;
                ent[k] = vertex_entry<kTab, kFlushProbes>(
                    v, owner[k], [&](int e, int32_t id) { return atomicCAS(&keys[e], -1, id); });
            }
#pragma unroll
            for (int k = 0; k < 2; k++) {
                if (ent[k] < 0) continue;
#pragma unroll
                for (int c = 0; c < 7; c++) lds_add_f64(&sums[7 * ent[k] + c], acc[7 * k + c]);
            }
            // The entries are listed compactly; then eight lanes per entry add its seven sums to the vertex's
            // 32-byte row of the interleaved accumulator, one wave instruction per eight vertices.
            int32_t* list = reinterpret_cast<int32_t*>(&A.val[0]);  // free after the rounds: 256 words
            const uint64_t own0 = ballot(owner[0]), own1 = ballot(owner[1]);
            const uint32_t n0 = (uint32_t)popc64(own0), nown = n0 + (uint32_t)popc64(own1);
            if (owner[0]) list[popc64(own0 & lanemask_lt())] = ent[0];
            if (owner[1]) list[n0 + popc64(own1 & lanemask_lt())] = ent[1];
            __syncthreads();
            // The next batch's vertex data is requested before the atomics, so staging it does not wait for them.
            // Only lanes 0..31 hold that batch's record words (of a part: lanes 0 to its count).
            nd = RecordData{};  // or its old values would be live, and spilled, throughout the batch
            if (more && lane < (kPart ? nnxt : kBatch)) fetch_record_data<kCell>(pos, col, nxt, nd);
            uint32_t issued = 0;
            {
                const int c = lane & 7;
                for (uint32_t b0 = 0; b0 < nown; b0 += 8) {
                    const uint32_t li = b0 + (uint32_t)(lane >> 3);
                    if (li < nown && c < 7) {
                        const int e = list[li];
                        const float val = (float)sums[7 * e + c];
                        if (val != 0.f) {
                            atomic_add_f32(&vacc[8 * (int64_t)keys[e] + c], val);
                            issued++;
                        }
                    }
                }
            }
#pragma unroll
            for (int k = 0; k < 2; k++) {
                // a slot that found no entry issues its own values
                if (!slot_live || ent[k] >= 0) continue;
                const int64_t g = k == 0 ? v0 : v1;
#pragma unroll
                for (int c = 0; c < 7; c++) {
                    const float val = acc[7 * k + c];
                    if (val == 0.f) continue;
                    issued++;
                    atomic_add_f32(&vacc[8 * g + c], val);
                }
            }
            natom += issued;
        }
        if (ballot(!done) == 0ull) break;
        __syncthreads();
    }
    if (ps.counters != nullptr) {
        const uint32_t tot = wave_inclusive_scan(natom);
        if (lane == 63 && tot) atomicAdd(ps.counters, (unsigned long long)tot);
    }
}

// Waves per SIMD that the registers allow: 3 for the exact adjoint (168 VGPRs of the 512 per lane; its 13,312 B of LDS
// fit 11 times, not 12), 2 for the reference one, whose sub-segment arrays need more of both.  kQueue as in
// k_render_forward.
template <bool kRef, bool kCell, bool kSub, bool kQueue>
__global__ __launch_bounds__(64, kRef ? 2 : 3) void k_render_adjoint(const BatchItem* __restrict__ items,
                                                        const AdjointTarget* __restrict__ targets, int nitems,
                                                        const uint32_t* __restrict__ order,
                                                        RecordStream stream,
                                                        const uint2* __restrict__ ranges, PixelState ps_all,
                                                        int use_abs, uint32_t* __restrict__ queue,
                                                        uint32_t ntiles) {
    __shared__ RecordVidLds L;
    __shared__ AdjFragLds A;
    __shared__ float4 s_seg[kRef ? 3 : 1][kRoundAdj];  // reference mode: sub-segment colours, then their adjoints
    if constexpr (!kQueue) {
        adjoint_tile<kRef, kCell, kSub>(items, targets, nitems, stream, ranges, ps_all, use_abs,
                                        global_tile_of_block(order), L, A, s_seg);
    } else {
        for (uint32_t t = claim_tile(queue); t < ntiles; t = claim_tile(queue)) {
            adjoint_tile<kRef, kCell, kSub>(items, targets, nitems, stream, ranges, ps_all, use_abs,
                                            order != nullptr ? order[t] : t, L, A, s_seg);
            __syncthreads();
        }
    }
}

template <bool kRef, bool kCell, int kEdge>
__global__ __launch_bounds__(64, kRef ? 2 : 3) void k_render_adjoint_parts(const BatchItem* __restrict__ items,
                                                                           const AdjointTarget* __restrict__ targets,
                                                                           int nitems,
                                                                           RecordStream stream,
                                                                           const uint2* __restrict__ ranges,
                                                                           PixelState ps_all, int use_abs) {
    __shared__ RecordVidLds L;
    __shared__ AdjFragLds A;
    __shared__ float4 s_seg[kRef ? 3 : 1][kRoundAdj];
    constexpr uint32_t kParts = PartOfTile<kEdge>::kParts;
    adjoint_tile<kRef, kCell, false, kEdge>(items, targets, nitems, stream, ranges, ps_all, use_abs,
                                            blockIdx.x / kParts, L, A, s_seg, blockIdx.x % kParts);
}

// Ordered fragment export (tet*4 + face per covered record), up to max_per_pixel per pixel.  It needs the records' ids
// and coverage only (kSub: and their faces' vertices, to test the coverage of the 8x8 sub-tile); a batch's record words
// are loaded a batch ahead, their indices two.
template <bool kSub>
__global__ __launch_bounds__(64) void k_export_fragments(const BatchItem* __restrict__ items, int nitems,
                                                          RecordStream stream,
                                                          const uint2* __restrict__ ranges, PixelState ps_all,
                                                          int max_per_pixel, int32_t* __restrict__ out_ids_all) {
    __shared__ RecordLds L;
    __shared__ int32_t s_stash[kSub ? 6 * kBatch : 1];
    const uint32_t gsub = global_tile_of_block(nullptr);
    const BatchItem& B = items[item_of_sub(items, nitems, gsub)];
    const ViewUniforms& U = B.U;
    const uint4* __restrict__ recs = stream.recs;
    const uint32_t* __restrict__ rec_of = stream.route->vals;
    const PixelState ps = item_pixel_state(ps_all, B);
    int32_t* __restrict__ out_ids = out_ids_all + B.pixel0 * max_per_pixel;
    const SubTile st = sub_tile(B, gsub);
    const int lane = threadIdx.x;
    const int lx = lane & 7, ly = lane >> 3;
    const int x = st.x0 + lx, y = st.y0 + ly;
    const bool valid = x < U.width && y < U.height;
    const uint2 rg = ranges[st.gtile];
    const int pix = valid ? pixel_index(U, x, y) : 0;
    const uint32_t last = valid ? ps.last_rec[pix] : 0u;
    int k = 0;
    RecordIn cur;
    uint32_t ahead = 0u;
    if (lane < kBatch && rg.x + lane < rg.y) cur = load_record(recs, rec_of[rg.x + lane]);
    if (lane < kBatch && rg.x + kBatch + lane < rg.y) ahead = rec_of[rg.x + kBatch + lane];
    for (uint32_t base = rg.x; base < rg.y; base += kBatch) {
        const int cnt = (int)min((uint32_t)kBatch, rg.y - base);
        if (lane < cnt) {
            if constexpr (kSub) {
                RecordData d;
                fetch_record_data(B.pos, nullptr, cur, d);
                store_record<true>(U, cur, d, L, lane, s_stash);
            } else {
                L.mask[0][lane] = cur.rec.y;
                L.mask[1][lane] = cur.rec.z;
            }
            L.meta[lane] = cur.rec.x;
        }
        if (lane < kBatch && base + kBatch + lane < rg.y) cur = load_record(recs, ahead);
        if (lane < kBatch && base + 2 * kBatch + lane < rg.y) ahead = rec_of[base + 2 * kBatch + lane];
        __syncthreads();
        if constexpr (kSub) {
            subtile_masks(L, s_stash, cnt, x, y, valid, lane);
            __syncthreads();
        }
        uint32_t m = valid ? lane_coverage(L, cnt, lane) : 0u;
        while (m) {
            const int j = __ffs(m) - 1;
            m &= m - 1u;
            if (base + j >= last) break;
            if (k < max_per_pixel) out_ids[(int64_t)pix * max_per_pixel + k] = (int32_t)L.meta[j];
            k++;
        }
        __syncthreads();
    }
    if (valid)
        for (; k < max_per_pixel; k++) out_ids[(int64_t)pix * max_per_pixel + k] = -1;
}

// Workgroups of `kernel` the GPU holds at once (the size of a persistent launch), computed once per kernel and
// device.
static unsigned resident_groups(const void* kernel) {
    static std::mutex mu;
    static std::map<std::pair<const void*, int>, unsigned> cache;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    std::lock_guard<std::mutex> lock(mu);
    auto it = cache.find({kernel, dev});
    if (it != cache.end()) return it->second;
    int per_cu = 0, cus = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, 64, 0) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
        return 0;
    const unsigned n = (unsigned)(per_cu > 0 ? per_cu : 1) * (unsigned)(cus > 0 ? cus : 1);
    cache[{kernel, dev}] = n;
    return n;
}

// One launch of a tile kernel: a workgroup per tile, or (queue != NULL) a persistent grid whose workgroups claim
// tiles from the queue counter, zeroed here first (a fill kernel, so that the launch can be graph-captured).
template <typename Kernel, typename... Args>
static void launch_tiles(Kernel grid_kernel, Kernel queue_kernel, int64_t ntiles, uint32_t* queue, hipStream_t s,
                         Args... args) {
    if (queue == nullptr) {
        hipLaunchKernelGGL(grid_kernel, dim3((unsigned)ntiles), dim3(64), 0, s, args..., queue, (uint32_t)ntiles);
        return;
    }
    unsigned grid = resident_groups(reinterpret_cast<const void*>(queue_kernel));
    if (grid == 0 || grid > (uint64_t)ntiles) grid = (unsigned)ntiles;
    fill_u32(queue, 0u, 1, s);
    hipLaunchKernelGGL(queue_kernel, dim3(grid), dim3(64), 0, s, args..., queue, (uint32_t)ntiles);
}

template <bool kCell, bool kSub, int kRound>
static void launch_forward_round(const BatchItem* items, int nitems, int64_t ntiles, const uint32_t* order,
                                 RecordStream recs, const uint2* ranges, PixelState ps, uint32_t* queue,
                                 hipStream_t s) {
    launch_tiles(k_render_forward<kCell, kRound, kSub, false>, k_render_forward<kCell, kRound, kSub, true>, ntiles,
                 queue, s, items, nitems, order, recs, ranges, ps);
}

template <bool kCell, bool kSub>
static void launch_forward_kind(const BatchItem* items, int nitems, int64_t ntiles, const uint32_t* order,
                                RecordStream recs, const uint2* ranges, PixelState ps, int round, uint32_t* queue,
                                hipStream_t s) {
    if (round == 64)
        launch_forward_round<kCell, kSub, 64>(items, nitems, ntiles, order, recs, ranges, ps, queue, s);
    else if (round == 256)
        launch_forward_round<kCell, kSub, 256>(items, nitems, ntiles, order, recs, ranges, ps, queue, s);
    else
        launch_forward_round<kCell, kSub, kRoundDefault>(items, nitems, ntiles, order, recs, ranges, ps, queue, s);
}

template <int kEdge>
static void launch_forward_parts(const BatchItem* items, int nitems, int64_t ntiles, RecordStream recs,
                                 const uint2* ranges, PixelState ps, uint32_t colour_kinds, hipStream_t s) {
    const dim3 grid((unsigned)(ntiles * PartOfTile<kEdge>::kParts));
    if (colour_kinds & kColoursPerVertex)
        hipLaunchKernelGGL((k_render_forward_parts<false, kEdge>), grid, dim3(64), 0, s, items, nitems, recs, ranges, ps);
    if (colour_kinds & kColoursPerCell)
        hipLaunchKernelGGL((k_render_forward_parts<true, kEdge>), grid, dim3(64), 0, s, items, nitems, recs, ranges, ps);
}

void launch_render_forward(const BatchItem* items, int nitems, int64_t ntiles, const uint32_t* order,
                           RecordStream recs, const uint2* ranges, PixelState ps, uint32_t colour_kinds,
                           hipStream_t s, int round, bool sub, uint32_t* queue, int edge) {
    if (ntiles <= 0) return;
    if (edge == 4) return launch_forward_parts<4>(items, nitems, ntiles, recs, ranges, ps, colour_kinds, s);
    if (edge == 2) return launch_forward_parts<2>(items, nitems, ntiles, recs, ranges, ps, colour_kinds, s);
    if (colour_kinds & kColoursPerVertex) {
        if (sub)
            launch_forward_kind<false, true>(items, nitems, ntiles, order, recs, ranges, ps, round, queue, s);
        else
            launch_forward_kind<false, false>(items, nitems, ntiles, order, recs, ranges, ps, round, queue, s);
    }
    if (colour_kinds & kColoursPerCell) {
        if (sub)
            launch_forward_kind<true, true>(items, nitems, ntiles, order, recs, ranges, ps, round, queue, s);
        else
            launch_forward_kind<true, false>(items, nitems, ntiles, order, recs, ranges, ps, round, queue, s);
    }
}

template <bool kRef, bool kCell, bool kSub>
static void launch_adjoint_kind(const BatchItem* items, const AdjointTarget* targets, int nitems, int64_t ntiles,
                                const uint32_t* order, RecordStream recs, const uint2* ranges, PixelState ps,
                                int use_abs, uint32_t* queue, hipStream_t s) {
    launch_tiles(k_render_adjoint<kRef, kCell, kSub, false>, k_render_adjoint<kRef, kCell, kSub, true>, ntiles,
                 queue, s, items, targets, nitems, order, recs, ranges, ps, use_abs);
}

template <bool kSub>
static void launch_adjoint_sub(const BatchItem* items, const AdjointTarget* targets, int nitems, int64_t ntiles,
                               const uint32_t* order, RecordStream recs, const uint2* ranges, PixelState ps,
                               int use_abs, int mode, uint32_t colour_kinds, uint32_t* queue, hipStream_t s) {
    if (colour_kinds & kColoursPerVertex) {
        if (mode == 1)
            launch_adjoint_kind<true, false, kSub>(items, targets, nitems, ntiles, order, recs, ranges, ps, use_abs,
                                                   queue, s);
        else
            launch_adjoint_kind<false, false, kSub>(items, targets, nitems, ntiles, order, recs, ranges, ps, use_abs,
                                                    queue, s);
    }
    if (colour_kinds & kColoursPerCell)  // exact adjoint only (the caller rejects mode 1 for such items)
        launch_adjoint_kind<false, true, kSub>(items, targets, nitems, ntiles, order, recs, ranges, ps, use_abs,
                                               queue, s);
}

template <int kEdge>
static void launch_adjoint_parts(const BatchItem* items, const AdjointTarget* targets, int nitems, int64_t ntiles,
                                 RecordStream recs, const uint2* ranges, PixelState ps, int use_abs, int mode,
                                 uint32_t colour_kinds, hipStream_t s) {
    const dim3 grid((unsigned)(ntiles * PartOfTile<kEdge>::kParts));
    if ((colour_kinds & kColoursPerVertex) && mode == 1)
        hipLaunchKernelGGL((k_render_adjoint_parts<true, false, kEdge>), grid, dim3(64), 0, s, items, targets, nitems,
                           recs, ranges, ps, use_abs);
    if ((colour_kinds & kColoursPerVertex) && mode != 1)
        hipLaunchKernelGGL((k_render_adjoint_parts<false, false, kEdge>), grid, dim3(64), 0, s, items, targets,
                           nitems, recs, ranges, ps, use_abs);
    if (colour_kinds & kColoursPerCell)
        hipLaunchKernelGGL((k_render_adjoint_parts<false, true, kEdge>), grid, dim3(64), 0, s, items, targets, nitems,
                           recs, ranges, ps, use_abs);
}

void launch_render_adjoint(const BatchItem* items, const AdjointTarget* targets, int nitems, int64_t ntiles,
                           const uint32_t* order, RecordStream recs, const uint2* ranges, PixelState ps, int use_abs,
                           int mode, uint32_t colour_kinds, hipStream_t s, bool sub, uint32_t* queue, int edge) {
    if (ntiles <= 0) return;
    if (edge == 4)
        return launch_adjoint_parts<4>(items, targets, nitems, ntiles, recs, ranges, ps, use_abs, mode, colour_kinds,
                                       s);
    if (edge == 2)
        return launch_adjoint_parts<2>(items, targets, nitems, ntiles, recs, ranges, ps, use_abs, mode, colour_kinds,
                                       s);
    if (sub)
        launch_adjoint_sub<true>(items, targets, nitems, ntiles, order, recs, ranges, ps, use_abs, mode,
                                 colour_kinds, queue, s);
    else
        launch_adjoint_sub<false>(items, targets, nitems, ntiles, order, recs, ranges, ps, use_abs, mode,
                                  colour_kinds, queue, s);
}

// Up to kFolds meshes' folds in one launch: each is less work than a launch of its own costs (a batched step of five small
// Delaunay balls 879 -> 871 us).
constexpr int kFolds = 8;
struct FoldList {
    VertexFold fold[kFolds];
    uint32_t block0[kFolds];  // first workgroup of each
    int n;
};

// grad_pos[v] += acc[v][0..2], grad_col[v] += acc[v][3..6].  One thread per vertex, so plain read-modify-writes.
__global__ __launch_bounds__(256) void k_fold_vertex_grads(FoldList list) {
    int k = 0;
#pragma unroll
    for (int i = 1; i < kFolds; i++) k = i < list.n && blockIdx.x >= list.block0[i] ? i : k;
    const VertexFold f = list.fold[k];
    const int64_t v = (int64_t)(blockIdx.x - list.block0[k]) * 256 + threadIdx.x;
    if (v >= f.V) return;
    const float4* __restrict__ acc = reinterpret_cast<const float4*>(f.acc);
    const float4 a = acc[2 * v], b = acc[2 * v + 1];
    f.grad_pos[3 * v + 0] += a.x;
    f.grad_pos[3 * v + 1] += a.y;
    f.grad_pos[3 * v + 2] += a.z;
    if (f.grad_col != nullptr) {
        f.grad_col[4 * v + 0] += a.w;
        f.grad_col[4 * v + 1] += b.x;
        f.grad_col[4 * v + 2] += b.y;
        f.grad_col[4 * v + 3] += b.z;
    }
}

// Whether two folds write to a common float: such folds run one after the other.
static bool folds_overlap(const VertexFold& a, const VertexFold& b) {
    const float* at[2] = {a.grad_pos, a.grad_col};
    const float* bt[2] = {b.grad_pos, b.grad_col};
    for (int i = 0; i < 2; i++)
        for (int j = 0; j < 2; j++) {
            if (at[i] == nullptr || bt[j] == nullptr) continue;
            const uintptr_t a0 = (uintptr_t)at[i], a1 = a0 + 4u * (uintptr_t)((3 + i) * a.V);
            const uintptr_t b0 = (uintptr_t)bt[j], b1 = b0 + 4u * (uintptr_t)((3 + j) * b.V);
            if (a0 < b1 && b0 < a1) return true;
        }
    return false;
}

void launch_fold_vertex_grads(const VertexFold* folds, int n, hipStream_t s) {
    FoldList list;
    uint32_t blocks = 0;
    list.n = 0;
    auto flush = [&] {
        if (list.n > 0) hipLaunchKernelGGL(k_fold_vertex_grads, dim3(blocks), dim3(256), 0, s, list);
        list.n = 0;
        blocks = 0;
    };
    for (int i = 0; i < n; i++) {
        if (folds[i].V <= 0) continue;
        bool apart = list.n == kFolds;
        for (int k = 0; k < list.n && !apart; k++) apart = folds_overlap(list.fold[k], folds[i]);
        if (apart) flush();
        list.fold[list.n] = folds[i];
        list.block0[list.n++] = blocks;
        blocks += (uint32_t)((folds[i].V + 255) / 256);
    }
    flush();
}

void launch_export_fragments(const BatchItem* items, int nitems, int64_t ntiles, RecordStream recs,
                             const uint2* ranges, PixelState ps, bool sub, int max_per_pixel, int32_t* out_ids,
                             hipStream_t s) {
    if (ntiles <= 0) return;
    const auto kernel = sub ? k_export_fragments<true> : k_export_fragments<false>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)ntiles), dim3(64), 0, s,
                       items, nitems, recs, ranges, ps, max_per_pixel, out_ids);
}

}  // namespace dtv
