// Fixed-point screen-tile rasterisation shared by the binning passes of the tile renderers: tile ranges of a
// screen triangle, the per-tile reject test and the exact 8x8 pixel-centre coverage (the tie rule gives each
// shared edge to exactly one side).
#pragma once
#include "dtv_device.h"
#include "dtv_prims.h"

namespace dtv {

struct FaceBins {
    int32_t tx0, tx1, ty0, ty1;  // tile range of the face's pixel-centre bounding box (empty: tx0 > tx1)
    int32_t shift;               // log2 of the tile edge in pixels (3, 4 or 5)
};

// Tile range of screen triangle S (its pixel-centre bounding box, clipped to the view).
__device__ __forceinline__ FaceBins screen_bins(const ViewUniforms& U, const ScreenTri& S) {
    FaceBins b;
    b.tx0 = 0;
    b.tx1 = -1;
    b.ty0 = 0;
    b.ty1 = -1;
    b.shift = U.tile_shift;
    int32_t x0, x1, y0, y1;
    tri_pixel_bbox(U, S, x0, x1, y0, y1);
    if (x0 > x1 || y0 > y1) return b;
    b.tx0 = x0 >> b.shift;
    b.tx1 = x1 >> b.shift;
    b.ty0 = y0 >> b.shift;
    b.ty1 = y1 >> b.shift;
    return b;
}

// Edge e of the oriented screen triangle: E(px, py) = dx (py - Y_a) - dy (px - X_a) in 1/256-pixel units; a
// pixel centre is inside when every E > 0, or E == 0 on a tie edge (dy < 0, or dy == 0 and dx > 0).
struct TileEdge {
    long long C;       // E at the centre of the tile's first pixel
    long long sx, sy;  // change of E per pixel step in x and y
    bool tie;
};

// (tx, ty): a tile of 1 << shift pixels.
__device__ __forceinline__ TileEdge tile_edge(const ScreenTri& S, int e, int tx, int ty, int shift) {
    const int a = e, b = e == 2 ? 0 : e + 1;
    const long long dx = S.X[b] - S.X[a], dy = S.Y[b] - S.Y[a];
    const long long px0 = 256LL * ((long long)tx << shift) + 128, py0 = 256LL * ((long long)ty << shift) + 128;
    TileEdge t;
    t.C = dx * (py0 - S.Y[a]) - dy * (px0 - S.X[a]);
    t.sx = -dy * 256;
    t.sy = dx * 256;
    t.tie = dy < 0 || (dy == 0 && dx > 0);
    return t;
}
// False when some edge function is negative at every pixel centre of tile (tx, ty): a record of that tile
// could not cover a pixel.  (The maximum of E over the tile's centre lattice sits at a corner.)
__device__ __forceinline__ bool tile_may_cover(const ScreenTri& S, int tx, int ty, int shift) {
    const long long n1 = (1 << shift) - 1;
#pragma unroll
    for (int e = 0; e < 3; e++) {
        const TileEdge t = tile_edge(S, e, tx, ty, shift);
        const long long mx = t.C + (t.sx > 0 ? n1 * t.sx : 0) + (t.sy > 0 ? n1 * t.sy : 0);
        if (mx < 0) return false;
    }
    return true;
}

// Pixel (x, y)'s centre inside oriented screen triangle (X, Y): every edge function E > 0, or E == 0 on a tie
// edge; the rule of tile_coverage, for one pixel.
__device__ __forceinline__ bool pixel_inside(const int32_t X[3], const int32_t Y[3], int x, int y) {
    const long long px = 256LL * x + 128, py = 256LL * y + 128;
    bool in = true;
#pragma unroll
    for (int e = 0; e < 3; e++) {
        const int a = e, b = e == 2 ? 0 : e + 1;
        const long long dx = (long long)X[b] - X[a], dy = (long long)Y[b] - Y[a];
        const long long E = dx * (py - Y[a]) - dy * (px - X[a]);
        const bool tie = dy < 0 || (dy == 0 && dx > 0);
        in = in && (E > 0 || (E == 0 && tie));
    }
    return in;
}

// Binning tiles larger than 8x8: a face whose bounding box spans more tiles than this keeps every tile of it, untested;
// the renderers test the coverage per pixel, so the records beyond the face cover nothing.
constexpr int kMaxTestedTiles = 64;

// Exact coverage of 8x8 tile (tx, ty): bit ly * 8 + lx is set when the centre of pixel (8 tx + lx, 8 ty + ly) is
// inside the triangle; pixels outside the viewport are clear.
//
// Per edge E = 256 W + r with W = q + ly dx - lx dy, q = floor(C / 256), r = C mod 256 (C: E at the tile's first
// pixel), so E > 0, or E == 0 on a tie edge  <=>  W >= wmin.  Screen coordinates span less than 2^26 (the guard band
// of 16 viewports, 1/256 pixel), so ly dx - lx dy stays below 7 * 2^27 < 2^30 in magnitude and q may be clamped to
// +-2^30, beyond which it decides every pixel: all of it is exact in 32 bits.  The three edges' signs are combined
// per pixel and collected by one funnel shift, 5 instructions a pixel without branches.
__device__ __forceinline__ uint64_t tile_coverage(const ScreenTri& S, int tx, int ty, int width, int height) {
    const int32_t px = 2048 * tx + 128, py = 2048 * ty + 128;
    int32_t dx[3], dy[3], row[3];  // row: W - wmin at the last pixel of the row in hand
#pragma unroll
    for (int e = 0; e < 3; e++) {
        const int a = e, b = e == 2 ? 0 : e + 1;
        dx[e] = S.X[b] - S.X[a];
        dy[e] = S.Y[b] - S.Y[a];
        const int64_t C = (int64_t)dx[e] * (int64_t)(py - S.Y[a]) - (int64_t)dy[e] * (int64_t)(px - S.X[a]);
        const int32_t hi = (int32_t)(C >> 38);
        int32_t q = (int32_t)(C >> 8);
        q = hi > 0 ? (1 << 30) : hi < -1 ? -(1 << 30) : q;
        const bool tie = dy[e] < 0 || (dy[e] == 0 && dx[e] > 0);
        const int32_t wmin = ((uint32_t)C & 255u) != 0u || tie ? 0 : 1;
        row[e] = (q - wmin) + 7 * (dx[e] - dy[e]);
    }
    uint32_t out[2];
#pragma unroll
    for (int half = 1; half >= 0; half--) {
        uint32_t m = 0u;  // sign bits, first pixel highest: set outside
#pragma unroll
        for (int ly = 3; ly >= 0; ly--) {
            int32_t v[3] = {row[0], row[1], row[2]};
#pragma unroll
            for (int lx = 7; lx >= 0; lx--) {
                m = __builtin_amdgcn_alignbit(m, (uint32_t)(v[0] | v[1] | v[2]), 31u);
#pragma unroll
                for (int e = 0; e < 3; e++) v[e] += dy[e];
            }
#pragma unroll
            for (int e = 0; e < 3; e++) row[e] -= dx[e];
        }
        out[half] = ~m;
    }
    const int nx = min(8, width - 8 * tx), ny = min(8, height - 8 * ty);
    uint64_t m = ((uint64_t)out[1] << 32) | out[0];
    if (nx < 8) m &= 0x0101010101010101ull * ((1ull << nx) - 1ull);
    if (ny < 8) m &= (1ull << (8 * ny)) - 1ull;
    return m;
}

__device__ __forceinline__ uint32_t wave_sum_u32(uint32_t v) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
    return v;
}
}  // namespace dtv
