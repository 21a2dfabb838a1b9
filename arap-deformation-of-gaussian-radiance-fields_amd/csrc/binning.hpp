// Tile lists of a render (binning.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "common.hpp"

namespace arapgs {

// Tiles of a record: id of the rectangle's first tile (over all views) in the
// high half and its width in the low half of base_w, and its number of tiles.
struct TileRect {
    uint32_t base_w;
    uint32_t area;
};
// Tile ids of this path fit 16 bits, and so does the width of a rectangle (one row
// of all 65,536 tiles takes the other path).
constexpr int64_t BIN_MAX_TILES = 65536;

struct BinInput {
    int64_t records;       // (view, Gaussian) records, at most 2^31 - 1
    int64_t visible;       // those with a tile
    uint32_t instances;    // their tiles in all, at most 2^31 - 1
    const float* depth;    // per record; 0 where nothing is visible
    const TileRect* rects; // per record; read where visible
    uint32_t dmin;         // smallest depth bits of the visible records
    int dbits;             // bits of (largest - smallest + 1)
    int gx;                // tiles per row of a view
    int64_t tiles;         // of all views, at most BIN_MAX_TILES
};

size_t bin_record_bytes(int64_t records);
size_t bin_instance_bytes(int64_t instances);
// *vals (in inst_ws) = the record of every instance, ordered by (tile, depth
// bits, record); ranges[t] = the [begin, end) of tile t.
int launch_binning(const BinInput& in, void* rec_ws, void* inst_ws, const uint32_t** vals, uint2* ranges,
                   hipStream_t st);

}  // namespace arapgs
