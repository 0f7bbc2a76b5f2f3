// Host-side launchers of the difftetvr_amd kernels (internal; the public surface is include/difftetvr_amd.h).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <string>

#include "dtv_device.h"

namespace dtv {

// sort.hip
void fill_u32(uint32_t* p, uint32_t v, int64_t n, hipStream_t s);
// Zeroes up to kClearRegions word ranges in one launch; a non-NULL item_dst also receives *item, and a non-NULL
// targets_dst the ntargets (<= kClearTargets) targets, all carried as kernel arguments (no host staging).
constexpr int kClearRegions = 6, kClearTargets = 8;
struct ClearList {
    uint32_t* p[kClearRegions];
    int64_t n[kClearRegions];  // words
    int count = 0;
    void add(void* ptr, int64_t words) {
        p[count] = static_cast<uint32_t*>(ptr);
        n[count++] = words;
    }
};
void launch_clear(const ClearList& regions, const BatchItem* item, BatchItem* item_dst, const AdjointTarget* targets,
                  int ntargets, AdjointTarget* targets_dst, hipStream_t s);

// What one render keeps in a small device buffer.  The words up to `cleared` are zeroed before binning.
constexpr int kBinSlots = 64;
struct BinSlot {
    uint32_t tris;     // visible faces (Projection: triangles)
    uint32_t not_min;  // complement of the smallest depth key
    uint32_t max;      // largest depth key
    uint32_t pad;
};
// Where the sort left its result (written by its histogram kernel).
struct SortRoute {
    const uint32_t* keys;  // sorted compact keys; tile_of_key(key, tile_shift)
    const uint32_t* vals;  // sorted record indices
    uint2* masks;          // room for one coverage mask per sorted record
    uint32_t tile_shift;
};
struct ViewScratch {
    BinSlot slots[kBinSlots];
    uint64_t total;     // records, written or not
    uint32_t ticket;
    uint32_t overflow;  // a record lay beyond the capacity
    uint32_t cleared;   // (marks the end of the zeroed words)
    uint32_t queue;     // tile work queue
    unsigned long long atomics;
    SortRoute route;
};

// The records' sort: by tile, then depth key, equal keys in record order.
struct SortInput {
    uint64_t* keys;  // [cap] tile << 32 | depth key; overwritten
    uint64_t* keys2; // [cap]
    uint32_t* vals;  // [cap]
    uint32_t* vals2; // [cap]
    int64_t cap;             // records the launches are sized for
    const uint64_t* n_dev;   // actual count in device memory, clamped to cap; NULL: cap
    const BinSlot* slots;    // the depth keys' range in device memory, or NULL: dmin and dbits below
    uint32_t dmin;           // smallest depth key
    int dbits;               // bits of the largest depth key minus dmin
    int tbits;               // bits of a tile number
};
int sort_bits(uint32_t range);       // bits of an unsigned number
int sort_max_passes(int tbits);      // passes at most
int64_t sort_lookback_words(int64_t cap, int passes);
// hist: [8 * 256] words and counters: [8] words, zeroed by the caller; lookback: sort_lookback_words.  Returns the
// passes launched.
int sort_records(const SortInput& in, uint32_t* hist, uint32_t* counters, uint32_t* lookback, SortRoute* route,
                 hipStream_t s);

// binning.hip
int64_t bin_blocks(int64_t T);  // 256-tet blocks
int64_t bin_status_words(int64_t nblocks);  // look-back words (64 bits) of a launch
bool bin_small(int64_t tets, int64_t pixels);  // whether workgroups of 64 tets are faster than ones of 256
struct BinOut {
    uint64_t* status;      // [bin_status_words(blocks)] look-back words, zeroed
    ViewScratch* scratch;
    uint64_t* keys;        // [cap] tile << 32 | depth key
    uint4* recs;           // [cap] records: two uint4 each (Projection: one)
    uint64_t cap;
};
// Bins the tets of all items (item i owns blocks [block0_i, block0_{i+1}) of 256 tets): scratch->total records, of
// which those below cap are written, in (tet, face, tile) order.
void launch_bin(const BatchItem* items, int nitems, int64_t nblocks, bool small, const BinOut& out, hipStream_t s);
// ranges[t] (zeroed): the sorted records of tile t.  recs (may be NULL): the unsorted records, rec_len uint4 each,
// whose coverage masks then go to route->masks in sorted order.
void launch_tile_ranges(const SortRoute* route, int64_t n, const uint64_t* n_dev, uint2* ranges, const uint4* recs,
                        int rec_len, hipStream_t s);
// cost[g] = record count of the binning tile holding 8x8 sub-tile g, for g < nsub.
void launch_subtile_cost(const BatchItem* items, int nitems, int64_t nsub, const uint2* ranges, uint32_t* cost,
                         hipStream_t s);
// Launch order of the tile renderers: order[0, num_tiles) lists every tile once, heaviest first, by the tile's
// cost: its record count (cost == NULL: ranges[t].y - ranges[t].x) or cost[t].  Costs are ranked in buckets of
// 1/8 octave; the order within a bucket is unspecified.  One workgroup; needs no cleared memory.
void launch_tile_order(const uint2* ranges, const uint32_t* cost, int64_t num_tiles, uint32_t* order,
                       hipStream_t s);

// render.hip
// The records in binning order (two uint4 each; Projection one) and the sort's result.
struct RecordStream {
    const uint4* recs;
    const SortRoute* route;
};
// Per-pixel state of a rendered batch, concatenated over its items (P = all pixels of the batch); item i's
// checkpoint planes start at max_ckpt * pixel0_i.
struct PixelState {
    float4* ray_color;      // [P] composite before the clear-colour blend: premultiplied RGB, transmittance
    uint32_t* frag_count;   // [P] fragments composited
    uint32_t* last_rec;     // [P] index (in the sorted record list) one past the last composited record
    uint32_t* num_ckpt;     // [P]
    float* ckpt_t;          // [max_ckpt][P] transmittance after ckpt_n fragments
    uint32_t* ckpt_n;       // [max_ckpt][P]
    unsigned long long* counters;  // optional (NULL): [0] += gradient float atomics issued by the adjoint
    uint32_t* tile_frags;   // [tiles of the batch] fragments composited per tile (written by the forward)
};
// ps.tile_frags from ps.frag_count (which a forward of parts of tiles does not write), for the batch's nsub sub-tiles.
void launch_tile_frags(const BatchItem* items, int nitems, int64_t nsub, PixelState ps, hipStream_t s);
// order (may be NULL = tile t in workgroup t): the tile each workgroup renders, from launch_tile_order.
// colour_kinds: which colour storages the batch's items use (kColoursPerVertex | kColoursPerCell); one launch
// per kind present, each rendering the tiles of its items.
constexpr uint32_t kColoursPerVertex = 1, kColoursPerCell = 2;
// round: fragments shaded per round of the forward (64, 128 or 256; other values take 128).  ntiles counts
// 8x8 sub-tiles (one workgroup each).
// sub: the batch bins tiles larger than 8x8 (the kernels then test coverage per 8x8 sub-tile).
// queue: NULL launches one workgroup per tile; else a persistent grid (the workgroups the GPU holds at once)
// takes the tiles in launch order from this device counter, which each launch zeroes first.
// recs: the records in binning order; the sorted order is route->vals.
// edge: 8, or 4 or 2 for (8 / edge)^2 waves per tile, each rendering edge x edge pixels (128 fragments per round,
// 8x8 binning tiles, no queue; order is not used).
void launch_render_forward(const BatchItem* items, int nitems, int64_t ntiles, const uint32_t* order,
                           RecordStream recs, const uint2* ranges, PixelState ps, uint32_t colour_kinds,
                           hipStream_t s, int round = 128, bool sub = false, uint32_t* queue = nullptr,
                           int edge = 8);
void launch_render_adjoint(const BatchItem* items, const AdjointTarget* targets, int nitems, int64_t ntiles,
                           const uint32_t* order, RecordStream recs, const uint2* ranges, PixelState ps, int use_abs,
                           int mode, uint32_t colour_kinds, hipStream_t s, bool sub = false,
                           uint32_t* queue = nullptr, int edge = 8);
// One mesh's interleaved gradient rows (8 floats per vertex: xyz, rgba) and the gradients they are added to (grad_col
// NULL: positions only).
struct VertexFold {
    const float* acc;
    int64_t V;
    float* grad_pos;
    float* grad_col;
};
// Adds the tile renderer adjoint's interleaved accumulator rows acc [V][8] of each fold into its grad_pos [V][3] and,
// unless NULL, grad_col [V][4].
void launch_fold_vertex_grads(const VertexFold* folds, int n, hipStream_t s);
void launch_export_fragments(const BatchItem* items, int nitems, int64_t ntiles, RecordStream recs,
                             const uint2* ranges, PixelState ps, bool sub, int max_per_pixel, int32_t* out_ids,
                             hipStream_t s);

// proj.hip: the Projection renderer.  Per-tet buffers are indexed by the tet's slot in the batch's block grid
// (block0 * 256 + tet): pt_info [slots], pt_vert / pt_col [5 * slots] (the five vertices' NDC xyz + thickness,
// colour); tri_grad [21 * 4 * slots] (the adjoint's per-triangle-corner sums).  Records: recs[i] =
// {triangle slot id (tet * 4 + k, item-local tet), coverage mask low, high, corner slots}.
void launch_pt_bin(const BatchItem* items, int nitems, int64_t nblocks, uint32_t* pt_info, float4* pt_vert,
                   float4* pt_col, bool small, const BinOut& out, hipStream_t s);
// edge: 8, or 4 for four waves per tile, each rendering 4x4 pixels (order is then not used).
void launch_pt_forward(const BatchItem* items, int nitems, int64_t ntiles, const uint32_t* order,
                       const float4* pt_vert, const float4* pt_col, RecordStream recs, const uint2* ranges,
                       PixelState ps, int edge, hipStream_t s);
void launch_pt_adjoint(const BatchItem* items, const AdjointTarget* targets, int nitems, int64_t ntiles,
                       int64_t nblocks, const uint32_t* order, const uint32_t* pt_info, const float4* pt_vert,
                       const float4* pt_col, RecordStream recs, const uint2* ranges, PixelState ps, float* tri_grad,
                       int64_t tri_grad_floats, int use_abs, int edge, hipStream_t s);

// optim.hip
struct AdamGroupDev {
    float* param;
    float* grad;
    float* m;
    float* v;
    int64_t n;
    float step_size;    // lr / (1 - beta1^t)
    float bc2_sqrt;     // sqrt(1 - beta2^t)
    float w1;           // 1 - beta1
    float beta2;
    float w2;           // 1 - beta2
    float eps;
    int32_t clamp_nonneg;
    int32_t zero_grad;
    double lr, beta1, beta2d;  // for bias corrections computed on the device
};
// step_dev (may be NULL): steps taken so far in device memory; then the bias corrections use step_dev + 1
// (step_size / bc2_sqrt of the groups are ignored) and a second launch increments it.
void launch_adam(const AdamGroupDev* groups, int ngroups, int64_t* step_dev, hipStream_t s);
void launch_mse(const float* img, const float* tgt, int64_t n, int64_t denom, float* dimg, float* loss,
                hipStream_t s);

// regularizer.hip
// V: the mesh's vertices (a rule of the launch looks at how many tets share one).
void launch_tet_regularizer(const int32_t* cells, const float* pos, int64_t T, int64_t V, float lambda, float beta,
                            float* grad_pos, hipStream_t s);

// api.hip: sets the message dtv_last_error() returns and passes the status code through.
int report_error(int code, const std::string& msg);

}  // namespace dtv
