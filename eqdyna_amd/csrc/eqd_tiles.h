// Tiles of the regular elements (host side): compact groups of at most
// kTileElems elements, one workgroup of elem_regular_kernel each, so that the
// workgroup can sum and update the nodes that no other element touches.
#pragma once
#include <cstdint>
#include <vector>

#include "eqd_device.h"

namespace eqd {

// Regular elements from which on a scenario runs in tiles.  Below about three
// tiles per CU a launch is one chain of waits, which the barrier and the
// nodes' loads lengthen: chunks of steps of 90,192 elements (dipping fault,
// FP64) 10.07 -> 10.84 ms with tiles; 167,808 (plastic) 11.38 -> 10.54,
// 200,000 (uniform, FP64) 14.94 -> 15.05, 686,000 (rough fault, FP64)
// 55.4 -> 51.2, 2.17 M (layered with Q, FP32) 96.7 -> 91.9, 2.42 M (rough
// fault, FP32) 214.1 -> 212.
constexpr int64_t kTileMinElems = 131072;

struct TileSet {
    std::vector<Tile> tile;
    std::vector<uint16_t> node_ent;  // 8 per inner node, tile by tile: staged forces in ascending element order
                                     // (kTileNone: none)
    std::vector<uint16_t> slot_src;  // staged force that fills each slot (kTileNone: padding)
    std::vector<uint32_t> slot_of;   // [8 n] slot of element t's force on local node a at t * 8 + a (kEntNone: inner)
    std::vector<uint8_t> inner;      // [nn] 1: the node is an inner node of a tile
    // order of the nodes on the device: node n of the reference at at[n], ref its inverse
    std::vector<int32_t> at, ref;
    int64_t n_inner;
};

// Order ids (elements of one class, 0-based, ascending) tile by tile and
// describe the tiles.  ien: 8 one-based nodes per element; degree: element
// entries of every node over all classes; outer[n] != 0 keeps node n out of
// the inner nodes.  Returns false, with ids as they were, when the elements do
// not group into well filled tiles.
bool make_tiles(std::vector<int32_t> &ids, const int32_t *ien, int64_t nn, const std::vector<int32_t> &degree,
                const std::vector<uint8_t> &outer, TileSet &T);

}  // namespace eqd
