// Tiles of the elements: grid positions from the connectivity, a tile shape for
// the grid's size, and per tile the inner nodes, their force entries
// and the slots of the forces that leave the tile.
#include "eqd_tiles.h"

#include <algorithm>
#include <array>
#include <cstdlib>
#include <numeric>

namespace eqd {

namespace {

typedef std::array<int32_t, 3> Pos;

// Integer grid positions of all elements, from element to element over shared
// corners: the neighbour in local direction d of an element is the one whose
// node 0 is the element's node at the other end of its edge in that direction.
// Elements are met in their given order, in which one of a grid's neighbours
// comes before each but the first.  Any positions are valid (they only decide
// which elements run together); comp numbers the connected pieces as they are
// met.  Wedges (elements with a repeated node), whose edges do not follow the
// grid, stay out: comp -1.  Returns the number of pieces.
int32_t grid_positions(const int32_t *ien, int64_t ne, int64_t nn, std::vector<Pos> &pos, std::vector<int32_t> &comp)
{
    constexpr int end[3] = {1, 3, 4};  // local node at the far end of node 0's edge in each direction
    std::vector<int32_t> own[4];       // element whose local node 0, 1, 3, 4 is the node
    constexpr int at[4] = {0, 1, 3, 4};
    pos.assign((size_t)ne, Pos{0, 0, 0});
    comp.assign((size_t)ne, -2);  // not met yet
#pragma omp parallel for schedule(static)
    for (int64_t e = 0; e < ne; e++) {
        const int32_t *nd = ien + e * 8;
        for (int a = 0; a < 8; a++)
            for (int b = 0; b < a; b++)
                if (nd[a] == nd[b]) comp[e] = -1;
    }
#pragma omp parallel for schedule(static, 1)
    for (int k = 0; k < 4; k++) {
        own[k].assign((size_t)nn, -1);
        for (int64_t e = 0; e < ne; e++)
            if (comp[e] != -1) own[k][ien[e * 8 + at[k]] - 1] = (int32_t)e;
    }
    int32_t ncomp = 0;
    for (int64_t e = 0; e < ne; e++) {
        if (comp[e] == -1) continue;
        const int32_t *nd = ien + e * 8;
        for (int d = 0; d < 3 && comp[e] < 0; d++)
            for (int ahead = 0; ahead < 2; ahead++) {
                const int32_t u = ahead ? own[0][nd[end[d]] - 1] : own[d + 1][nd[0] - 1];
                if (u < 0 || comp[u] < 0) continue;
                comp[e] = comp[u];
                pos[e] = pos[u];
                pos[e][d] += ahead ? -1 : 1;
                break;
            }
        if (comp[e] < 0) comp[e] = ncomp++;
    }
    return ncomp;
}

// Tiles along each direction for a grid of N elements: the box of at most
// kTileElems elements that leaves the most nodes inside the tiles, less what
// its unfilled lanes cost.
void tile_counts(const int64_t N[3], int64_t cnt[3])
{
    double best = -1e300;
    for (int x = 3; x <= 16; x++)
        for (int y = 3; y <= 16; y++)
            for (int z = 3; z <= 16; z++) {
                if (x * y * z > kTileElems) continue;
                const int64_t c[3] = {(N[0] + x - 1) / x, (N[1] + y - 1) / y, (N[2] + z - 1) / z};
                const double n = (double)N[0] * N[1] * N[2];
                const double in = (double)(N[0] - c[0]) * (N[1] - c[1]) * (N[2] - c[2]) / n;
                const double fill = n / ((double)c[0] * c[1] * c[2] * kTileElems);
                const double score = in + 0.5 * fill;
                if (score > best) {
                    best = score;
                    std::copy(c, c + 3, cnt);
                }
            }
}

struct Grid {
    std::vector<Pos> pos;
    std::vector<int32_t> part;  // [ne] 27 * piece + which third in each direction, -1 a wedge
    int32_t parts;
    int fast;  // direction in which node numbers run
};

// Pieces and, in each direction, the thirds below, beside and above the regular
// elements: the PML elements then fall into layers, edges and corners that
// are boxes of their own, whatever the layers' thickness.
bool make_grid(const std::vector<int32_t> &reg, const int32_t *ien, int64_t ne, int64_t nn, Grid &G)
{
    const int32_t ncomp = grid_positions(ien, ne, nn, G.pos, G.part);
    if (ncomp > 1000) return false;
    std::vector<Pos> lo((size_t)ncomp, Pos{INT32_MAX, INT32_MAX, INT32_MAX}),
        hi((size_t)ncomp, Pos{INT32_MIN, INT32_MIN, INT32_MIN});
    for (int32_t e : reg)
        for (int d = 0; d < 3 && G.part[e] >= 0; d++) {
            lo[G.part[e]][d] = std::min(lo[G.part[e]][d], G.pos[e][d]);
            hi[G.part[e]][d] = std::max(hi[G.part[e]][d], G.pos[e][d]);
        }
#pragma omp parallel for schedule(static)
    for (int64_t e = 0; e < ne; e++) {
        const int32_t c = G.part[e];
        if (c < 0) continue;
        int third = 0;
        for (int d = 0; d < 3; d++) third = third * 3 + (G.pos[e][d] < lo[c][d] ? 0 : G.pos[e][d] > hi[c][d] ? 2 : 1);
        G.part[e] = c * 27 + third;
    }
    G.parts = ncomp * 27;
    const int32_t *nd = ien + ne / 2 * 8;
    const int step[3] = {std::abs(nd[1] - nd[0]), std::abs(nd[3] - nd[0]), std::abs(nd[4] - nd[0])};
    G.fast = 0;
    for (int d = 1; d < 3; d++)
        if (step[d] < step[G.fast]) G.fast = d;
    return true;
}

// ids tile by tile; false, with ids as they were, when they do not fill their tiles
bool group(std::vector<int32_t> &ids, const Grid &G, double min_fill, std::vector<Tile> &tile)
{
    const int64_t n = (int64_t)ids.size();
    std::vector<Pos> lo((size_t)G.parts, Pos{INT32_MAX, INT32_MAX, INT32_MAX}),
        hi((size_t)G.parts, Pos{INT32_MIN, INT32_MIN, INT32_MIN});
    int64_t nwedge = 0;
    for (int32_t e : ids) {
        const int32_t c = G.part[e];
        if (c < 0) nwedge++;
        for (int d = 0; d < 3 && c >= 0; d++) {
            lo[c][d] = std::min(lo[c][d], G.pos[e][d]);
            hi[c][d] = std::max(hi[c][d], G.pos[e][d]);
        }
    }
    const int fast = G.fast, o1 = (fast + 1) % 3, o2 = (fast + 2) % 3;
    std::vector<std::array<int64_t, 3>> cnt((size_t)G.parts), len((size_t)G.parts);
    std::vector<int64_t> base((size_t)G.parts + 1, 0);
    for (int32_t c = 0; c < G.parts; c++) {
        base[c + 1] = base[c];
        if (lo[c][0] > hi[c][0]) continue;  // no element of the class
        for (int d = 0; d < 3; d++) len[c][d] = (int64_t)hi[c][d] - lo[c][d] + 1;
        tile_counts(len[c].data(), cnt[c].data());
        base[c + 1] += cnt[c][0] * cnt[c][1] * cnt[c][2];
        if (base[c + 1] > 4 * n + 64) return false;
    }
    // elements by box, and within a box in rows along the fast direction;
    // wedges in their given order, in boxes of their own
    const int64_t nbox = base[G.parts] + (nwedge + kTileElems - 1) / kTileElems;
    std::vector<int32_t> box((size_t)n);
    std::vector<int64_t> start((size_t)nbox + 1, 0);
    int64_t w = 0;
    for (int64_t t = 0; t < n; t++) {
        const int32_t c = G.part[ids[t]];
        if (c < 0) {
            box[t] = (int32_t)(base[G.parts] + w++ / kTileElems);
        } else {
            int64_t b[3];
            for (int d = 0; d < 3; d++) b[d] = (int64_t)(G.pos[ids[t]][d] - lo[c][d]) * cnt[c][d] / len[c][d];
            box[t] = (int32_t)(base[c] + (b[o2] * cnt[c][o1] + b[o1]) * cnt[c][fast] + b[fast]);
        }
        start[box[t] + 1]++;
    }
    int64_t ntile = 0;
    for (int64_t b = 0; b < nbox; b++) ntile += (start[b + 1] + kTileElems - 1) / kTileElems;
    // lanes without an element cost their share of every workgroup
    if ((double)n < min_fill * (double)(ntile * kTileElems)) return false;
    if (!slots_fit(n, ntile)) return false;
    std::partial_sum(start.begin(), start.end(), start.begin());
    std::vector<int32_t> out((size_t)n);
    {
        std::vector<int64_t> at(start.begin(), start.end() - 1);
        for (int64_t t = 0; t < n; t++) out[at[box[t]]++] = ids[t];
    }
#pragma omp parallel for schedule(dynamic, 64)
    for (int64_t b = 0; b < nbox; b++)
        std::sort(out.begin() + start[b], out.begin() + start[b + 1], [&](int32_t x, int32_t y) {
            const Pos &p = G.pos[x], &q = G.pos[y];
            if (p[o2] != q[o2]) return p[o2] < q[o2];
            if (p[o1] != q[o1]) return p[o1] < q[o1];
            if (p[fast] != q[fast]) return p[fast] < q[fast];
            return x < y;
        });
    for (int64_t b = 0; b < nbox; b++)
        for (int64_t e = start[b]; e < start[b + 1]; e += kTileElems)
            tile.push_back(Tile{(int32_t)e, (int32_t)std::min<int64_t>(kTileElems, start[b + 1] - e), 0, 0, 0, 0, 0});
    ids.swap(out);
    return true;
}

}  // namespace

bool make_tiles(std::vector<int32_t> *const ids[2], const bool want[2], const int32_t *ien, int64_t ne, int64_t nn,
                const std::vector<int32_t> &degree, const std::vector<uint8_t> &kind, double min_fill, TileSet T[2],
                NodeOrder &O)
{
    if (!want[0] && !want[1]) return false;
    Grid G;
    if (!make_grid(*ids[0], ien, ne, nn, G)) return false;
    for (int c = 0; c < 2; c++)
        if (want[c] && !ids[c]->empty()) group(*ids[c], G, min_fill, T[c].tile);
    const int64_t nt0 = (int64_t)T[0].tile.size(), nt = nt0 + (int64_t)T[1].tile.size();
    if (nt == 0) return false;
    auto tile = [&](int64_t k) -> Tile & { return k < nt0 ? T[0].tile[k] : T[1].tile[k - nt0]; };
    // The first and last tile that touches a node; nodes in the order of their
    // first tile, a tile's inner nodes first and then its others by last tile,
    // so that a tile's inner nodes, and the nodes that the same tiles share,
    // are neighbours in memory.  Nodes of no tile come first.
    std::vector<int32_t> first((size_t)nn, -1), last((size_t)nn, -1), touch((size_t)nn, 0);
    auto lower = [](int32_t &x, int32_t v) {
        int32_t c = __atomic_load_n(&x, __ATOMIC_RELAXED);
        while ((c < 0 || v < c) && !__atomic_compare_exchange_n(&x, &c, v, true, __ATOMIC_RELAXED, __ATOMIC_RELAXED)) {}
    };
    auto raise = [](int32_t &x, int32_t v) {
        int32_t c = __atomic_load_n(&x, __ATOMIC_RELAXED);
        while (v > c && !__atomic_compare_exchange_n(&x, &c, v, true, __ATOMIC_RELAXED, __ATOMIC_RELAXED)) {}
    };
#pragma omp parallel for schedule(dynamic, 64)
    for (int64_t k = 0; k < nt; k++) {
        const Tile &K = tile(k);
        const std::vector<int32_t> &el = *ids[k < nt0 ? 0 : 1];
        for (int32_t t = K.e0; t < K.e0 + K.ne; t++)
            for (int a = 0; a < 8; a++) {
                const int32_t nd = ien[(int64_t)el[t] * 8 + a] - 1;
                lower(first[nd], (int32_t)k);
                raise(last[nd], (int32_t)k);
                __atomic_fetch_add(&touch[nd], 1, __ATOMIC_RELAXED);
            }
    }
    auto own = [&](int32_t nd) {
        return first[nd] >= 0 && first[nd] == last[nd] && touch[nd] == degree[nd] && degree[nd] <= 8 &&
               kind[nd] == (first[nd] < nt0 ? 1 : 2);
    };
    std::vector<int64_t> nstart((size_t)nt + 2, 0);
    for (int64_t n = 0; n < nn; n++) nstart[first[n] + 2]++;
    std::partial_sum(nstart.begin(), nstart.end(), nstart.begin());
    O.ref.resize((size_t)nn);
    O.at.resize((size_t)nn);
    {
        std::vector<int64_t> at(nstart.begin(), nstart.end() - 1);
        for (int64_t n = 0; n < nn; n++) O.ref[at[first[n] + 1]++] = (int32_t)n;
    }
#pragma omp parallel for schedule(dynamic, 64)
    for (int64_t k = 0; k < nt; k++) {
        const auto b = O.ref.begin() + nstart[k + 1], e = O.ref.begin() + nstart[k + 2];
        // A workgroup updates one node a thread.  Tiles among other elements own
        // fewer nodes than elements, but one at free faces on opposite sides (a
        // slab of any extent, or a mesh of one tile) owns up to
        // (x + 1)(y + 1)(z + 1): those past the workgroup stay with the node kernels.
        auto mid = std::stable_partition(b, e, [&](int32_t n) { return own(n); });
        if (mid - b > kTileElems) mid = b + kTileElems;
        std::stable_sort(mid, e, [&](int32_t x, int32_t y) { return last[x] < last[y]; });
        tile(k).n0 = (int32_t)nstart[k + 1];
        tile(k).nn = (int32_t)(mid - b);
    }
    O.inner.assign((size_t)nn, 0);
#pragma omp parallel for schedule(static)
    for (int64_t i = 0; i < nn; i++) O.at[O.ref[i]] = (int32_t)i;
#pragma omp parallel for schedule(static)
    for (int64_t k = 0; k < nt; k++)
        for (int32_t i = tile(k).n0; i < tile(k).n0 + tile(k).nn; i++) O.inner[O.ref[i]] = 1;
    // per tile: its (node, element, local node) entries in the order a node
    // sums them; an inner node's become its row of node_ent, the others slots
    // in runs of neighbouring nodes' q-th entries, as the node kernels read them
    // (an entry as one number: node, the element's rank in its tile, local node, lane)
    auto node_of = [](uint64_t e) { return (int32_t)(e >> 24); };
    auto src_of = [](uint64_t e) { return (uint16_t)((e >> 8 & 7) * kTileElems + (e & 255)); };
    static_assert(kTileElems == 256, "lane and rank are 8 bits");
    for (int c = 0; c < 2; c++) {
        TileSet &S = T[c];
        const std::vector<int32_t> &el = *ids[c];
        const int64_t ntc = (int64_t)S.tile.size();
        if (ntc == 0) continue;
        S.slot_of.assign(el.size() * 8, kEntNone);
        for (Tile &K : S.tile) {
            K.i0 = (int32_t)S.n_inner;
            S.n_inner += K.nn;
        }
        S.node_ent.assign((size_t)S.n_inner * 8, kTileNone);
        std::vector<std::vector<uint16_t>> tsrc((size_t)ntc);
#pragma omp parallel
        {
            std::vector<uint64_t> E;
            std::vector<std::pair<int32_t, uint16_t>> B;  // q and source of a run's entries
            std::vector<int32_t> byid;
#pragma omp for schedule(dynamic, 16)
            for (int64_t k = 0; k < ntc; k++) {
                const Tile &K = S.tile[k];
                byid.assign(el.begin() + K.e0, el.begin() + K.e0 + K.ne);
                std::sort(byid.begin(), byid.end());
                E.clear();
                for (int l = 0; l < K.ne; l++) {
                    const int32_t e = el[K.e0 + l];
                    const uint64_t rank = std::lower_bound(byid.begin(), byid.end(), e) - byid.begin();
                    for (int a = 0; a < 8; a++)
                        E.push_back((uint64_t)O.at[ien[(int64_t)e * 8 + a] - 1] << 24 | rank << 16 | (uint64_t)a << 8 | l);
                }
                std::sort(E.begin(), E.end());
                // the other nodes in runs that the same tiles share: such nodes follow
                // one another
                auto flush = [&] {
                    for (int32_t q = 0; !B.empty(); q++) {
                        size_t left = 0;
                        for (const auto &x : B) {
                            if (x.first == q) tsrc[k].push_back(x.second);
                            else B[left++] = x;
                        }
                        B.resize(left);
                    }
                };
                int32_t f = -1, g = -1;
                for (size_t i = 0; i < E.size();) {
                    const int32_t nd = node_of(E[i]), rn = O.ref[nd];
                    const bool in = O.inner[rn] != 0;
                    if (!in && (first[rn] != f || last[rn] != g)) {
                        flush();
                        f = first[rn];
                        g = last[rn];
                    }
                    for (int32_t q = 0; i < E.size() && node_of(E[i]) == nd; i++, q++) {
                        if (in) S.node_ent[((int64_t)K.i0 + nd - K.n0) * 8 + q] = src_of(E[i]);
                        else B.push_back({q, src_of(E[i])});
                    }
                }
                flush();
                tsrc[k].resize((tsrc[k].size() + 63) / 64 * 64, kTileNone);
            }
        }
        int64_t slots = 0;
        for (int64_t k = 0; k < ntc; k++) {
            S.tile[k].s0 = (int32_t)(slots / 64);
            S.tile[k].ns = (int32_t)tsrc[k].size();
            slots += S.tile[k].ns;
        }
        S.slot_src.resize((size_t)slots);
#pragma omp parallel for schedule(static)
        for (int64_t k = 0; k < ntc; k++) {
            const Tile &K = S.tile[k];
            const int64_t s0 = (int64_t)K.s0 * 64;
            for (int i = 0; i < K.ns; i++) {
                const uint16_t src = tsrc[k][i];
                S.slot_src[s0 + i] = src;
                if (src != kTileNone)
                    S.slot_of[((int64_t)K.e0 + src % kTileElems) * 8 + src / kTileElems] = (uint32_t)(s0 + i);
            }
        }
    }
    return true;
}

}  // namespace eqd
