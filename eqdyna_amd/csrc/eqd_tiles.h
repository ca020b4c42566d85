// Tiles of the elements (host side): compact groups of at most kTileElems
// elements of a class, one workgroup of its element kernel each, so that the
// workgroup can sum and update the nodes that no other element touches.
#pragma once
#include <cstdint>
#include <vector>

#include "eqd_device.h"

namespace eqd {

// Regular elements from which on a scenario runs in tiles.  Below about three
// tiles per CU a launch is one chain of waits, which the barrier and the
// nodes' loads lengthen, and elements without tiles share a launch with the
// PML elements.  Step without tiles and with them: 148,000 elements (rough
// fault, FP64) 112.2 and 121.9 us, FP32 74.0 and 75.6; 167,808 (plastic) 102.1
// and 86.8, 200,000 (uniform, FP64) 115.9 and 101.2; chunks of 150 to 400 steps
// of 686,000 (rough fault, FP64) 55.4 and 51.2 ms, 2.17 M (layered with Q, FP32)
// 96.7 and 91.9.
constexpr int64_t kTileMinElems = 163840;
// The same for the PML elements, whose tiles have three barriers: 127,932
// (plastic, FP64) neutral, ensembles of 130,000 at most (FP32) 22.1 -> 23.9 ms
// with tiles, 232,000 (uniform, FP64) 15.03 -> 13.37, 466,000 (rough fault,
// FP64) 51.2 -> 47.6, 938,200 (layered, FP32) 91.6 -> 89.9, 1.04 M (rough fault,
// FP32) 200.4 -> 192.3.
constexpr int64_t kTileMinPml = 196608;
// Share of the tiles' lanes that must hold an element.
constexpr double kTileMinFill = 0.625;

// whether any slot of n elements in ntile tiles has a number that an entry of the
// gather tables can hold: at most 8 slots an element, and each tile's are rounded up
// to 64
inline bool slots_fit(int64_t n, int64_t ntile) { return 8 * n + 64 * ntile < (int64_t)kEntSlotMask; }

// one class's tiles (none: tile is empty)
struct TileSet {
    std::vector<Tile> tile;
    std::vector<uint16_t> node_ent;  // 8 per inner node, tile by tile: staged forces in ascending element order
                                     // (kTileNone: none)
    std::vector<uint16_t> slot_src;  // staged force that fills each slot (kTileNone: padding)
    std::vector<uint32_t> slot_of;   // [8 n] slot of element t's force on local node a at t * 8 + a (kEntNone: inner)
    int64_t n_inner = 0;
};

// order of the nodes on the device: node n of the reference at at[n], ref its
// inverse; inner[n] 1 where the node is an inner node of a tile
struct NodeOrder {
    std::vector<int32_t> at, ref;
    std::vector<uint8_t> inner;
};

// Order ids[c] (elements of class c, 0 regular, 1 PML; 0-based, ascending)
// tile by tile for the classes that are wanted and fill their tiles to at least
// min_fill on average, describe their tiles in T[c] and order the nodes.  ien: 8 one-based
// nodes per element; degree: element entries of every node; kind[n]: the class
// whose tiles node n may be an inner node of, plus one (0: none).  Returns
// whether any class runs in tiles.
bool make_tiles(std::vector<int32_t> *const ids[2], const bool want[2], const int32_t *ien, int64_t ne, int64_t nn,
                const std::vector<int32_t> &degree, const std::vector<uint8_t> &kind, double min_fill, TileSet T[2],
                NodeOrder &O);

}  // namespace eqd
