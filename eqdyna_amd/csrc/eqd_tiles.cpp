// Tiles of the regular elements: grid positions from the connectivity, a tile
// shape for the grid's size, and per tile the inner nodes, their force entries
// and the slots of the forces that leave the tile.
#include "eqd_tiles.h"

#include <algorithm>
#include <array>
#include <cstdlib>
#include <numeric>

namespace eqd {

namespace {

typedef std::array<int32_t, 3> Pos;

// Integer grid positions of the elements, walking from element to element over
// shared corners: the neighbour in local direction d of an element is the one
// whose node 0 is the element's node at the other end of its edge in that
// direction.  Any positions are valid (they only decide which elements run
// together); comp numbers the connected pieces.  Wedges (elements with a
// repeated node), whose edges do not follow the grid, stay out: comp -1.
void grid_positions(const std::vector<int32_t> &ids, const int32_t *ien, int64_t nn, std::vector<Pos> &pos,
                    std::vector<int32_t> &comp, int32_t *ncomp)
{
    const int64_t n = (int64_t)ids.size();
    constexpr int end[3] = {1, 3, 4};  // local node at the far end of node 0's edge in each direction
    std::vector<int32_t> own[4];       // element whose local node 0, 1, 3, 4 is the node
    constexpr int at[4] = {0, 1, 3, 4};
    std::vector<uint8_t> wedge((size_t)n);
#pragma omp parallel for schedule(static)
    for (int64_t t = 0; t < n; t++) {
        const int32_t *nd = ien + (int64_t)ids[t] * 8;
        for (int a = 0; a < 8; a++)
            for (int b = 0; b < a; b++)
                if (nd[a] == nd[b]) wedge[t] = 1;
    }
#pragma omp parallel for schedule(static, 1)
    for (int k = 0; k < 4; k++) {
        own[k].assign((size_t)nn, -1);
        for (int64_t t = 0; t < n; t++)
            if (!wedge[t]) own[k][ien[(int64_t)ids[t] * 8 + at[k]] - 1] = (int32_t)t;
    }
    pos.assign((size_t)n, Pos{0, 0, 0});
    comp.assign((size_t)n, -1);
    std::vector<int32_t> stack;
    *ncomp = 0;
    for (int64_t s = 0; s < n; s++) {
        if (wedge[s] || comp[s] >= 0) continue;
        comp[s] = *ncomp;
        stack.push_back((int32_t)s);
        while (!stack.empty()) {
            const int32_t t = stack.back();
            stack.pop_back();
            const int32_t *nd = ien + (int64_t)ids[t] * 8;
            for (int d = 0; d < 3; d++)
                for (int back = 0; back < 2; back++) {
                    const int32_t u = back ? own[d + 1][nd[0] - 1] : own[0][nd[end[d]] - 1];
                    if (u < 0 || comp[u] >= 0) continue;
                    comp[u] = *ncomp;
                    pos[u] = pos[t];
                    pos[u][d] += back ? -1 : 1;
                    stack.push_back(u);
                }
        }
        ++*ncomp;
    }
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

}  // namespace

bool make_tiles(std::vector<int32_t> &ids, const int32_t *ien, int64_t nn, const std::vector<int32_t> &degree,
                const std::vector<uint8_t> &outer, TileSet &T)
{
    const int64_t n = (int64_t)ids.size();
    if (n == 0) return false;
    std::vector<Pos> pos;
    std::vector<int32_t> comp;
    int32_t ncomp;
    grid_positions(ids, ien, nn, pos, comp, &ncomp);
    std::vector<Pos> lo((size_t)ncomp, Pos{INT32_MAX, INT32_MAX, INT32_MAX}), hi((size_t)ncomp, Pos{INT32_MIN, INT32_MIN, INT32_MIN});
    for (int64_t t = 0; t < n; t++)
        for (int d = 0; d < 3 && comp[t] >= 0; d++) {
            lo[comp[t]][d] = std::min(lo[comp[t]][d], pos[t][d]);
            hi[comp[t]][d] = std::max(hi[comp[t]][d], pos[t][d]);
        }
    // the direction in which node numbers run, from a middle element
    int fast = 0;
    {
        const int32_t *nd = ien + (int64_t)ids[n / 2] * 8;
        const int step[3] = {std::abs(nd[1] - nd[0]), std::abs(nd[3] - nd[0]), std::abs(nd[4] - nd[0])};
        for (int d = 1; d < 3; d++)
            if (step[d] < step[fast]) fast = d;
    }
    const int o1 = (fast + 1) % 3, o2 = (fast + 2) % 3;
    std::vector<std::array<int64_t, 3>> cnt((size_t)ncomp), len((size_t)ncomp);
    std::vector<int64_t> base((size_t)ncomp + 1, 0);
    for (int32_t c = 0; c < ncomp; c++) {
        for (int d = 0; d < 3; d++) len[c][d] = (int64_t)hi[c][d] - lo[c][d] + 1;
        tile_counts(len[c].data(), cnt[c].data());
        base[c + 1] = base[c] + cnt[c][0] * cnt[c][1] * cnt[c][2];
        if (base[c + 1] > 4 * n) return false;
    }
    // elements by box, and within a box in rows along the fast direction
    const int64_t nwedge = std::count(comp.begin(), comp.end(), -1);
    const int64_t nbox = base[ncomp] + (nwedge + kTileElems - 1) / kTileElems;
    std::vector<int32_t> box((size_t)n);
    std::vector<int64_t> start((size_t)nbox + 1, 0);
    int64_t w = 0;  // wedges in their given order, in boxes of their own
    for (int64_t t = 0; t < n; t++) {
        const int32_t c = comp[t];
        if (c < 0) {
            box[t] = (int32_t)(base[ncomp] + w++ / kTileElems);
            start[box[t] + 1]++;
            continue;
        }
        int64_t b[3];
        for (int d = 0; d < 3; d++) b[d] = (int64_t)(pos[t][d] - lo[c][d]) * cnt[c][d] / len[c][d];
        box[t] = (int32_t)(base[c] + (b[o2] * cnt[c][o1] + b[o1]) * cnt[c][fast] + b[fast]);
        start[box[t] + 1]++;
    }
    int64_t ntile = 0;
    for (int64_t b = 0; b < nbox; b++) ntile += (start[b + 1] + kTileElems - 1) / kTileElems;
    // lanes without an element cost their share of every workgroup
    if (n < ntile * (kTileElems * 5 / 8)) return false;
    std::partial_sum(start.begin(), start.end(), start.begin());
    std::vector<int32_t> ord((size_t)n);
    {
        std::vector<int64_t> at(start.begin(), start.end() - 1);
        for (int64_t t = 0; t < n; t++) ord[at[box[t]]++] = (int32_t)t;
    }
#pragma omp parallel for schedule(dynamic, 64)
    for (int64_t b = 0; b < nbox; b++)
        std::sort(ord.begin() + start[b], ord.begin() + start[b + 1], [&](int32_t x, int32_t y) {
            const Pos &p = pos[x], &q = pos[y];
            if (p[o2] != q[o2]) return p[o2] < q[o2];
            if (p[o1] != q[o1]) return p[o1] < q[o1];
            if (p[fast] != q[fast]) return p[fast] < q[fast];
            return x < y;
        });
    T.tile.clear();
    for (int64_t b = 0; b < nbox; b++)
        for (int64_t e = start[b]; e < start[b + 1]; e += kTileElems)
            T.tile.push_back(Tile{(int32_t)e, (int32_t)std::min<int64_t>(kTileElems, start[b + 1] - e), 0, 0, 0, 0, 0});
    std::vector<int32_t> out((size_t)n);
    for (int64_t t = 0; t < n; t++) out[t] = ids[ord[t]];
    // The first and last tile that touches a node; nodes in the order of their
    // first tile, a tile's inner nodes first and then its others by last tile,
    // so that a tile's inner nodes, and the nodes that the same tiles share,
    // are neighbours in memory.  Nodes of no tile come first.
    const int64_t nt = (int64_t)T.tile.size();
    std::vector<int32_t> first((size_t)nn, -1), last((size_t)nn, -1), touch((size_t)nn, 0);
    for (int64_t k = 0; k < nt; k++)
        for (int32_t t = T.tile[k].e0; t < T.tile[k].e0 + T.tile[k].ne; t++)
            for (int a = 0; a < 8; a++) {
                const int32_t nd = ien[(int64_t)out[t] * 8 + a] - 1;
                if (first[nd] < 0) first[nd] = (int32_t)k;
                last[nd] = (int32_t)k;
                touch[nd]++;
            }
    auto inner = [&](int32_t nd) {
        return first[nd] >= 0 && first[nd] == last[nd] && touch[nd] == degree[nd] && degree[nd] <= 8 && !outer[nd];
    };
    std::vector<int64_t> nstart((size_t)nt + 2, 0);
    for (int64_t n = 0; n < nn; n++) nstart[first[n] + 2]++;
    std::partial_sum(nstart.begin(), nstart.end(), nstart.begin());
    T.ref.resize((size_t)nn);
    T.at.resize((size_t)nn);
    {
        std::vector<int64_t> at(nstart.begin(), nstart.end() - 1);
        for (int64_t n = 0; n < nn; n++) T.ref[at[first[n] + 1]++] = (int32_t)n;
    }
    T.n_inner = 0;
    int64_t nin = 0;
#pragma omp parallel for schedule(dynamic, 64) reduction(+ : nin)
    for (int64_t k = 0; k < nt; k++) {
        const auto b = T.ref.begin() + nstart[k + 1], e = T.ref.begin() + nstart[k + 2];
        const auto mid = std::stable_partition(b, e, [&](int32_t n) { return inner(n); });
        std::stable_sort(mid, e, [&](int32_t x, int32_t y) { return last[x] < last[y]; });
        T.tile[k].n0 = (int32_t)nstart[k + 1];
        T.tile[k].nn = (int32_t)(mid - b);
        nin += mid - b;
    }
    T.n_inner = nin;
    T.inner.assign((size_t)nn, 0);
#pragma omp parallel for schedule(static)
    for (int64_t i = 0; i < nn; i++) {
        T.at[T.ref[i]] = (int32_t)i;
        T.inner[T.ref[i]] = inner(T.ref[i]);
    }
    // per tile: its (node, element, local node) entries in the order a node
    // sums them; an inner node's become its row of node_ent, the others slots
    // in runs of neighbouring nodes' q-th entries, as the node kernels read them
    T.slot_of.assign((size_t)n * 8, kEntNone);
    struct Entry {
        int32_t node, elem, q;
        uint16_t src;  // staged force: local node * kTileElems + lane
    };
    int64_t nodes = 0;
    for (Tile &K : T.tile) {
        K.i0 = (int32_t)nodes;
        nodes += K.nn;
    }
    T.node_ent.assign((size_t)nodes * 8, kTileNone);
    std::vector<std::vector<uint16_t>> tsrc((size_t)nt);
#pragma omp parallel
    {
        std::vector<Entry> E, S;
#pragma omp for schedule(dynamic, 16)
        for (int64_t k = 0; k < nt; k++) {
            const Tile &K = T.tile[k];
            E.clear();
            S.clear();
            for (int l = 0; l < K.ne; l++) {
                const int32_t e = out[K.e0 + l];
                for (int a = 0; a < 8; a++)
                    E.push_back(Entry{T.at[ien[(int64_t)e * 8 + a] - 1], e, 0, (uint16_t)(a * kTileElems + l)});
            }
            std::sort(E.begin(), E.end(), [](const Entry &x, const Entry &y) {
                if (x.node != y.node) return x.node < y.node;
                if (x.elem != y.elem) return x.elem < y.elem;
                return x.src < y.src;
            });
            for (size_t i = 0; i < E.size();) {
                const int32_t nd = E[i].node;
                for (int32_t q = 0; i < E.size() && E[i].node == nd; i++, q++) {
                    if (T.inner[T.ref[nd]]) {
                        T.node_ent[((int64_t)K.i0 + nd - K.n0) * 8 + q] = E[i].src;
                    } else {
                        E[i].q = q;
                        S.push_back(E[i]);
                    }
                }
            }
            std::sort(S.begin(), S.end(), [&](const Entry &x, const Entry &y) {
                const int32_t a = T.ref[x.node], b = T.ref[y.node];
                if (first[a] != first[b]) return first[a] < first[b];
                if (last[a] != last[b]) return last[a] < last[b];
                if (x.q != y.q) return x.q < y.q;
                return x.node < y.node;
            });
            for (const Entry &x : S) tsrc[k].push_back(x.src);
            tsrc[k].resize((tsrc[k].size() + 63) / 64 * 64, kTileNone);
        }
    }
    int64_t slots = 0;
    for (int64_t k = 0; k < nt; k++) {
        Tile &K = T.tile[k];
        K.s0 = (int32_t)(slots / 64);
        K.ns = (int32_t)tsrc[k].size();
        slots += K.ns;
    }
    if (slots > (int64_t)kEntSlotMask) return false;
    T.slot_src.resize((size_t)slots);
#pragma omp parallel for schedule(static)
    for (int64_t k = 0; k < nt; k++) {
        const Tile &K = T.tile[k];
        const int64_t s0 = (int64_t)K.s0 * 64;
        for (int i = 0; i < K.ns; i++) {
            const uint16_t src = tsrc[k][i];
            T.slot_src[s0 + i] = src;
            if (src != kTileNone)
                T.slot_of[((int64_t)K.e0 + src % kTileElems) * 8 + src / kTileElems] = (uint32_t)(s0 + i);
        }
    }
    ids.swap(out);
    return true;
}

}  // namespace eqd
