// Tiled triangular sweeps: the rows of a system are cut into tiles (boxes of
// space, or ranges of the numbering; a batch's stacked systems into ranges), one
// workgroup per tile, and the values of a tile's rows live in its LDS. Further
// wavefronts of the workgroup copy values between the LDS and memory where other
// tiles need them.
//
// A dependency inside a tile is seen through LDS, 0.2-0.35 us after it was
// computed; only a dependency on another tile goes through memory, where a
// value is seen 1.0-1.3 us after it was computed (timelines of FP64 sweeps).
// The dependency chain of tril(A) follows the grid, so it crosses a tile
// boundary a few times per axis instead of once per level. The factor is used
// as it is (no merged stencils), every row sums its entries in the factor's
// order, and the forward and the backward sweep are one launch.
//
// Layout: tiles hold nearly equal row counts; tile b owns positions
// [b S, (b+1) S), S a multiple of 64, its rows in dependency-level order and
// then padding (empty rows). The tile's wavefronts take 64-row chunks in turn.
// A chunk's entries are stored in pairs, pair by pair (64 lanes side by side),
// padded to the chunk's widest row (a level's rows are sorted by their lower
// entries, so forward 31 % and backward 56 % of the entries are padding in an
// octree of 3.5 M rows in block colours). An entry names the LDS slot of its
// value: [0, S) the tile's rows, [S, S + H) values imported from other tiles
// ("halo"), S + H a slot that always holds zero (padding entries). A tile's halo
// entries lie side by side in memory, in the order its rows need them; the tile
// that computes a value stores it there, once per reading tile, so polling reads
// whole cache lines.
#pragma once

#include <cstdint>

namespace astg {

// Wavefronts of a tile: computing, importing, exporting. 12 computing ones keep
// the loads of 12 chunks in flight: with 8 of them and each wavefront's next
// chunk loaded ahead the FP64 sweeps take about as long on small systems and
// 15 % longer at 1800 rows a tile. 16 in all is the register file's limit.
constexpr int kTileWaves = 12;
constexpr int kTileImport = 2;
constexpr int kTileExport = 2;

// A system's state in the batched solves: 16 doubles (BatchSlot), looked at as
// the upper words of the doubles.
constexpr int kSysStride = 32;

// One direction of the tiled sweeps (forward: lower entries, backward: upper).
struct TileDir {
    const int* sell;       // per chunk: first entry pair (64 lanes each); nchunks + 1
    const uint32_t* slot;  // per entry pair: the slots of both, low half first
    const int* hstart;     // per position: first halo entry; one more at the end
    const int* xstart;     // per position: first export; one more at the end
    const uint16_t* xslot; // per export: slot of its row
    const int* xdest;      // per export: the halo entry it fills
};

struct TileView {
    TileDir d[2];
    const uint8_t* step;  // per position: the rank of its level among its chunk's levels
    const int* order;  // per position: row, -1 padding
    const int* sys;    // batched solves, per position: the row's system
    const int* sysDone;  // and per system, kSysStride apart: nonzero once it has finished
    const int* finished; // per tile: nonzero once a system with rows in it has
    int S;             // positions per tile
    int slots;         // LDS slots: S + H + 1
    int exports;       // room of the LDS export list
    long long* trace;  // per-row timeline (3 per row), null in normal runs
};

}  // namespace astg
