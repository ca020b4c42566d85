// make_tiles (eqdyna_amd/csrc/eqd_tiles.h) for tests/test_tiles.py: one call,
// and the arrays it made.
#include <cstring>

#include "../eqdyna_amd/csrc/eqd_tiles.cpp"

namespace {
eqd::TileSet g_tiles[2];
eqd::NodeOrder g_order;
std::vector<int32_t> g_ids[2];
}  // namespace

extern "C" {

// cls: class of each element (0 regular, 1 PML); kind, want, min_fill as make_tiles
int tiles_make(const int32_t *ien, const uint8_t *cls, int64_t ne, int64_t nn, const uint8_t *kind, int want_regular,
               int want_pml, double min_fill)
{
    std::vector<int32_t> degree((size_t)nn, 0);
    for (int c = 0; c < 2; c++) {
        g_tiles[c] = eqd::TileSet();
        g_ids[c].clear();
    }
    g_order = eqd::NodeOrder();
    for (int64_t e = 0; e < ne; e++) g_ids[cls[e]].push_back((int32_t)e);
    for (int64_t i = 0; i < 8 * ne; i++) degree[ien[i] - 1]++;
    std::vector<int32_t> *const ids[2] = {&g_ids[0], &g_ids[1]};
    const bool want[2] = {want_regular != 0, want_pml != 0};
    return eqd::make_tiles(ids, want, ien, ne, nn, degree, std::vector<uint8_t>(kind, kind + nn), min_fill, g_tiles,
                           g_order);
}

int tiles_slots_fit(int64_t n, int64_t ntile) { return eqd::slots_fit(n, ntile); }

// an array of class c (or of the node order) and its number of values
const void *tiles_get(int c, const char *what, int64_t *count)
{
    auto give = [&](const auto &v, int64_t width) {
        *count = (int64_t)v.size() * width;
        return (const void *)v.data();
    };
    const eqd::TileSet &T = g_tiles[c];
    if (!strcmp(what, "tile")) return give(T.tile, sizeof(eqd::Tile) / sizeof(int32_t));
    if (!strcmp(what, "node_ent")) return give(T.node_ent, 1);
    if (!strcmp(what, "slot_src")) return give(T.slot_src, 1);
    if (!strcmp(what, "slot_of")) return give(T.slot_of, 1);
    if (!strcmp(what, "ids")) return give(g_ids[c], 1);
    if (!strcmp(what, "at")) return give(g_order.at, 1);
    if (!strcmp(what, "ref")) return give(g_order.ref, 1);
    if (!strcmp(what, "inner")) return give(g_order.inner, 1);
    *count = -1;
    return nullptr;
}
}
