// rvs_inpaint.h -- workspace layout and launcher of the exact inpainting kernels.
#ifndef RVS_INPAINT_H
#define RVS_INPAINT_H

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stddef.h>

#include "rvs_kernels.h"

namespace rvs_k {

constexpr int kInpTile = 32;            // edge of the tiles the inpainting works on
constexpr int kHoleTileBlocks = 2048;   // persistent blocks of the passes over the hole tiles
constexpr int kInpMaskWords = kInpTile + 2;

// 32 x 32 pixel tiles along one side.
__host__ __device__ inline int inpaint_tiles(int n) { return (n + kInpTile - 1) / kInpTile; }

// Per-tile arrays are indexed by [view][tile row][tile column] of 32 x 32
// pixel tiles (a view's tiles start at its hole_base) and stored only for tiles
// with holes; px by global pixel (a view's pixels start at its px_base).
struct InpaintWS {
    uint32_t* count;  // tiles with holes (zeroed before the launch set)
    uint8_t* thole;   // 1 when the tile has a hole (every tile)
    int2* htiles;     // the tiles with holes and their views, in no particular order
    uint32_t* mask;   // [tile][34] not-known bits of the tile's 32 rows, of the row below it and
                      // (by row) of the column right of it; pixels outside the image count as not known
    unsigned long long* rowc;  // [tile][32] minimum key of each tile row, then of the row before the tile
    unsigned long long* colc;  // [tile][32] the same per column, of the row minima
    unsigned long long* cola;  // [tile][32] backward pass: of the column's own pixels
    unsigned long long* rmin;  // [tile] smallest of the tile's 32 row carries
    int2* px;         // holes: forward distance and source (pixel of the view)
    int ntiles;       // tiles of all views
    const uint8_t* rflags;  // raster tile flags of the views (bit 1: a hole or a deferred pixel), or
                            // null; a 32 x 32 tile whose raster tiles all lack bit 1 has no hole
};

// npx, ntiles: pixels and 32 x 32 pixel tiles of all views.
size_t inpaint_ws_bytes(size_t npx, size_t ntiles);
InpaintWS inpaint_ws_carve(void* base, size_t npx, size_t ntiles);
// Inpaints every view of the batch in place (views[v].color from
// views[v].quality); *ws.count must be 0.
hipError_t launch_inpaint(const ViewDesc* views, int nviews, int max_w, int max_h, const InpaintWS& ws,
                          int32_t* map_out, hipStream_t s);

}  // namespace rvs_k

#endif
