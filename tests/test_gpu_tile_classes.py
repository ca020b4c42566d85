"""Tiles as the sizes of the two classes of elements decide (163,840 regular,
196,608 PML elements): meshes of which one class runs in tiles beside the other
in the reference's order, and class tables that fit beside a tile's stage in
LDS or do not.  Against no tiles at all: the same bits."""
import numpy as np
import pytest

from eqdyna_amd import case as cases
from eqdyna_amd import mesh
from eqdyna_amd.solver import Solver
from test_gpu_engine import assert_same

KEYS = ["fric", "fnft", "velArr", "dispArr", "v1", "nodalForceArr", "stressArr", "OffFaultStGramSCEC"]


def with_waves(b):
    # a wave field that fades towards the absorbing layers; both nodes of a pair move together
    x = b["meshCoor"]
    u = (x - x.min(0)) / np.ptp(x, axis=0)
    three = np.flatnonzero(b["numOfDofPerNodeArr"] == 3)
    v = np.zeros_like(x)
    v[three] = (0.02 * np.prod(np.sin(np.pi * u[:, :2]) ** 4, axis=1) * u[:, 2])[three, None] * np.cos(
        x[three] @ (2.0e-3 * np.array([[1.3, -0.7, 0.9], [0.8, 1.1, -1.4], [-0.6, 0.5, 1.2]])).T + np.arange(3))
    b = dict(b)
    b["velArr"], b["v1"] = v, b["v1"].copy()
    b["v1"][b["eqNumIndexArr"][b["eqNumStartIndexLoc"][three][:, None] + np.arange(3)] - 1] = v[three]
    return b


def compare(b, sc, precision, tiled, tag, monkeypatch):
    """The default against the reference's order; returns the default's layout."""
    out, layout = [], None
    for order in (None, "0"):
        if order:
            monkeypatch.setenv("EQD_ELEMENT_ORDER", order)
        else:
            monkeypatch.delenv("EQD_ELEMENT_ORDER", raising=False)
        print(f"case {tag} {precision} order {order}", flush=True)
        s = Solver(b, sc, precision)
        info = s.layout_info()
        layout = layout or info
        assert {k for k in ("tiles", "tiles_pml") if info[k] > 0} == (tiled if order is None else set())
        s.run(5)
        s.run(6)
        out.append({k: s.get(k) for k in KEYS})
        s.close()
    assert_same(out[0], out[1], f"{tag} {precision}")
    return layout


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("classes", ["tables", "rows"])
@pytest.mark.parametrize("nx,ny,nz,npml,tiled", [(45, 23, 37, 7, "tiles"), (40, 18, 40, 12, "tiles_pml")])
def test_one_class_in_tiles(nx, ny, nz, npml, tiled, classes, precision, monkeypatch):
    b, sc = mesh.build_case(cases.box_sw(nx, nz, ny, 100.0, npml))
    monkeypatch.setenv("EQD_NO_OPERATOR_CLASSES", "1" if classes == "rows" else "0")
    monkeypatch.setenv("EQD_GEOM_OPS", "0")  # operators rebuilt in the kernels: test_gpu_tiles.py
    compare(with_waves(b), sc, precision, {tiled}, f"{nx} {ny} {nz} {classes}", monkeypatch)


@pytest.mark.gpu
@pytest.mark.parametrize("layers", [6, 16, 40, 70])
def test_class_tables_beside_the_stage(layers, monkeypatch):
    # an FP64 PML tile stages 61,440 bytes: class tables up to 4 KiB sit beside
    # them in LDS, larger ones stay in memory (above 16 KiB in any launch; the
    # regular tiles' 49,152 bytes leave room for those)
    c = cases.box_sw(30, 70, 19, 100.0, 12)
    c.nmat, c.n2mat = layers, 4
    c.mat = cases.layered_medium(5, n_layers=layers, max_depth=-c.zmin)
    c.mat[:-1, 0] = np.round(np.linspace(100.0, -c.zmin - 100.0, layers - 1) / 100.0) * 100.0
    c.roumax, c.vmaxPML = float(c.mat[:, 3].max()), float(c.mat[:, 1].max())
    b, sc = mesh.build_case(c)
    info = compare(with_waves(b), sc, "fp64", {"tiles", "tiles_pml"}, f"{layers} layers", monkeypatch)
    size = 8 * (35 * info["op_classes_pml"] + 32 * info["phi_classes_pml"])
    print(f"{layers} layers: class tables of the PML elements {size} bytes", flush=True)
    assert (size <= 4096, size <= 16384) == (layers < 10, layers < 50) and info["op_classes_pml"] > 0
