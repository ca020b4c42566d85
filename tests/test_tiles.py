"""Tiles of the elements (eqd_tiles.cpp), on the CPU: every node's forces reach
it exactly once and in ascending element order, whatever the mesh's faces are.
A tile's workgroup of 256 updates one inner node a thread, so a tile has at
most 256 of them; slabs with free faces on both sides, and meshes of one tile,
would give it more.  What runs on these tables is compared with the
reference's order in test_gpu_tiles.py."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from eqdyna_amd import build_lib

HERE = os.path.dirname(os.path.abspath(__file__))
TILE, NONE16, NONE32 = 256, 0xFFFF, 0xFFFFFFFF


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("tiles") / "libtiles.so")
    subprocess.run([build_lib.HIPCC, "-O2", "-std=c++17", f"--offload-arch={build_lib.ARCH}", "-fPIC", "-fopenmp",
                    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-Wno-unused-command-line-argument",
                    "-x", "hip", os.path.join(HERE, "tiles_host.cpp"), "-shared", "-o", out], check=True)
    L = C.CDLL(out)
    L.tiles_make.argtypes = [C.c_void_p, C.c_void_p, C.c_int64, C.c_int64, C.c_void_p, C.c_int, C.c_int, C.c_double]
    L.tiles_slots_fit.argtypes = [C.c_int64, C.c_int64]
    L.tiles_get.argtypes = [C.c_int, C.c_char_p, C.POINTER(C.c_int64)]
    L.tiles_get.restype = C.c_void_p
    return L


def get(L, c, what, dtype):
    n = C.c_int64()
    p = L.tiles_get(c, what.encode(), C.byref(n))
    assert n.value >= 0, what
    if n.value == 0:
        return np.zeros(0, dtype)
    return np.ctypeslib.as_array((C.c_byte * (n.value * np.dtype(dtype).itemsize)).from_address(p)).view(dtype).copy()


def grid(nx, ny, nz):
    """ien (one-based) of a box of elements, numbered z fastest as the case builder does."""
    node = np.arange((nx + 1) * (ny + 1) * (nz + 1)).reshape(nx + 1, ny + 1, nz + 1)
    c = [node[:-1, :-1, :-1], node[1:, :-1, :-1], node[1:, 1:, :-1], node[:-1, 1:, :-1],
         node[:-1, :-1, 1:], node[1:, :-1, 1:], node[1:, 1:, 1:], node[:-1, 1:, 1:]]
    return np.stack([a.ravel() for a in c], axis=1).astype(np.int32) + 1, node.size


def make(L, ien, nn, cls, kind, want=(1, 1), min_fill=0.0):
    ien, cls, kind = np.ascontiguousarray(ien), np.ascontiguousarray(cls), np.ascontiguousarray(kind)
    return L.tiles_make(ien.ctypes.data, cls.ctypes.data, len(ien), nn, kind.ctypes.data, *want, min_fill)


def check(L, ien, nn, cls, kind):
    """The tables against the mesh; returns the largest number of inner nodes of a tile."""
    inner = get(L, 0, "inner", np.uint8)
    at, ref = get(L, 0, "at", np.int32), get(L, 0, "ref", np.int32)
    assert np.array_equal(at[ref], np.arange(nn)) and len(ref) == nn
    owned, most = np.zeros(nn, int), 0
    for c in (0, 1):
        ids = get(L, c, "ids", np.int32)
        assert np.array_equal(np.sort(ids), np.flatnonzero(cls == c))
        tiles = get(L, c, "tile", np.int32).reshape(-1, 7)
        if len(tiles) == 0:
            assert np.array_equal(ids, np.flatnonzero(cls == c))
            continue
        e0, ne, n0, cnt, i0, s0, ns = tiles.T
        assert np.array_equal(e0, np.cumsum(ne) - ne) and ne.sum() == len(ids) and ne.max() <= TILE
        assert np.array_equal(i0, np.cumsum(cnt) - cnt)
        most = max(most, int(cnt.max()))
        tile_of = np.repeat(np.arange(len(tiles)), ne)  # of each element in tile order
        lane = np.arange(len(ids)) - e0[tile_of]
        # inner nodes: the row's entries are the node's forces in ascending element order
        own = np.concatenate([np.arange(a, a + k) for a, k in zip(n0, cnt)]).astype(int)
        np.add.at(owned, ref[own], 1)
        assert np.all(kind[ref[own]] == c + 1)
        row = get(L, c, "node_ent", np.uint16).astype(int).reshape(-1, 8)
        k = np.repeat(np.arange(len(tiles)), cnt)
        used = row != NONE16
        el = np.where(used, ids[np.minimum(e0[k][:, None] + row % TILE, len(ids) - 1)], np.iinfo(np.int32).max)
        assert np.all((row % TILE < ne[k][:, None]) | ~used)
        key = el.astype(np.int64) * 8 + np.where(used, row // TILE, 0)
        assert np.all(np.diff(key, axis=1)[used[:, 1:]] > 0)
        hit = ien[np.where(used, el, 0), np.where(used, row // TILE, 0)] - 1
        assert np.all((hit == ref[own][:, None]) | ~used)
        degree = np.bincount(ien.ravel() - 1, minlength=nn)
        assert np.array_equal(used.sum(1), degree[ref[own]])
        # all other forces: a slot each, which the tile fills with that force
        slot = get(L, c, "slot_of", np.uint32).astype(np.int64).reshape(-1, 8)
        src = get(L, c, "slot_src", np.uint16).astype(int)
        out = inner[ien[ids] - 1] == 0
        assert np.array_equal(slot != NONE32, out)
        assert len(np.unique(slot[out])) == out.sum() == np.count_nonzero(src != NONE16)
        t, a = np.nonzero(out)
        assert np.array_equal(src[slot[out]], a * TILE + lane[t])
        lo = s0[tile_of[t]].astype(np.int64) * 64
        assert np.all((slot[out] >= lo) & (slot[out] < lo + ns[tile_of[t]]))
    assert np.array_equal(owned, inner)  # each once, and no other node is left to a tile
    return most


# (elements along x, y, z; what a tile would own without the bound)
@pytest.mark.parametrize("size,over", [((8, 8, 4), True), ((4, 4, 4), False), ((6, 6, 200), True), ((40, 36, 4), True),
                                       ((3, 70, 70), True), ((24, 24, 24), False), ((300, 140, 4), True)])
@pytest.mark.parametrize("c", [0, 1])
def test_tiles_of_a_box_with_free_faces(lib, size, over, c):
    ien, nn = grid(*size)
    cls, kind = np.full(len(ien), c, np.uint8), np.full(nn, c + 1, np.uint8)
    assert make(lib, ien, nn, cls, kind) == 1
    most = check(lib, ien, nn, cls, kind)
    assert most == TILE if over else most <= TILE


@pytest.mark.parametrize("want", [(1, 1), (1, 0), (0, 1)])
def test_tiles_of_a_box_in_an_absorbing_shell(lib, want):
    # PML on five sides, fixed outer nodes, some nodes that no tile may own
    size, p = (30, 26, 22), 5
    ien, nn = grid(*size)
    at = np.stack(np.unravel_index(np.arange(len(ien)), size), axis=1)
    pml = ((at < p) | (at >= np.array(size) - p))
    pml[:, 2] = at[:, 2] < p
    cls = pml.any(1).astype(np.uint8)
    kind = np.ones(nn, np.uint8)
    xyz = np.stack(np.unravel_index(np.arange(nn), [s + 1 for s in size]), axis=1)
    kind[((xyz < p) | (xyz > np.array(size) - p))[:, :2].any(1) | (xyz[:, 2] < p)] = 2
    kind[((xyz == 0) | (xyz == np.array(size)))[:, :2].any(1) | (xyz[:, 2] == 0)] = 0
    kind[::97] = 0
    assert make(lib, ien, nn, cls, kind, want) == 1
    check(lib, ien, nn, cls, kind)
    for c in (0, 1):
        assert (len(get(lib, c, "tile", np.int32)) > 0) == bool(want[c])


def test_a_class_that_does_not_fill_its_tiles_keeps_its_order(lib):
    # PML elements strewn over the whole grid fill no box; the regular ones are a box
    ien, nn = grid(20, 20, 20)
    cls = np.zeros(len(ien), np.uint8)
    cls[::11] = 1
    kind = np.ones(nn, np.uint8)
    assert make(lib, ien, nn, cls, kind, min_fill=0.625) == 1
    assert len(get(lib, 0, "tile", np.int32)) > 0 and len(get(lib, 1, "tile", np.int32)) == 0
    check(lib, ien, nn, cls, kind)  # (ids of the other class: ascending, as they were)
    assert make(lib, ien, nn, cls, kind, (0, 1), 0.625) == 0
    assert np.array_equal(get(lib, 1, "ids", np.int32), np.flatnonzero(cls == 1))


def test_slot_numbers_fit_a_table_entry(lib):
    # an entry has 31 bits for the slot, one value of which means none; tiles
    # that hold few elements each take 64 slots for one, more than the elements do
    limit = 2**31 - 1
    for n, ntile in ((1, 1), (100_000_000, 1_000_000), (33_554_431, 0), (2**25, 2**25), (2**24, 2**25), (2**28, 8),
                     (2**28 - 9, 8), (2**28 - 65, 8)):
        assert lib.tiles_slots_fit(n, ntile) == (8 * n + 64 * ntile < limit)
    assert not lib.tiles_slots_fit(2**25, 2**25) and lib.tiles_slots_fit(2**25, 2**17)
