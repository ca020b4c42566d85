"""Meshes of which one class of elements runs in tiles and the other does not,
by the sizes that decide (163,840 regular, 196,608 PML elements): regular
elements' tiles beside PML elements in the reference's order, and the other way
round.  Against no tiles at all: the same bits."""
import numpy as np
import pytest

from eqdyna_amd import case as cases
from eqdyna_amd import mesh
from eqdyna_amd.solver import Solver
from test_gpu_engine import assert_same

KEYS = ["fric", "fnft", "velArr", "dispArr", "v1", "nodalForceArr", "stressArr", "OffFaultStGramSCEC"]


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("classes", ["tables", "rows"])
@pytest.mark.parametrize("nx,ny,nz,npml,tiled", [(45, 23, 37, 7, "tiles"), (40, 18, 40, 12, "tiles_pml")])
def test_one_class_in_tiles(nx, ny, nz, npml, tiled, classes, precision, monkeypatch):
    b, sc = mesh.build_case(cases.box_sw(nx, nz, ny, 100.0, npml))
    # a wave field that fades towards the absorbing layers; both nodes of a pair move together
    x = b["meshCoor"]
    u = (x - x.min(0)) / np.ptp(x, axis=0)
    three = np.flatnonzero(b["numOfDofPerNodeArr"] == 3)
    v = np.zeros_like(x)
    v[three] = (0.02 * np.prod(np.sin(np.pi * u[:, :2]) ** 4, axis=1) * u[:, 2])[three, None] * np.cos(
        x[three] @ (2.0e-3 * np.array([[1.3, -0.7, 0.9], [0.8, 1.1, -1.4], [-0.6, 0.5, 1.2]])).T + np.arange(3))
    b["velArr"], b["v1"] = v, b["v1"].copy()
    b["v1"][b["eqNumIndexArr"][b["eqNumStartIndexLoc"][three][:, None] + np.arange(3)] - 1] = v[three]
    monkeypatch.setenv("EQD_NO_OPERATOR_CLASSES", "1" if classes == "rows" else "0")
    monkeypatch.setenv("EQD_GEOM_OPS", "0")  # operators rebuilt in the kernels: test_gpu_tiles.py
    out = []
    for order in (None, "0"):
        if order:
            monkeypatch.setenv("EQD_ELEMENT_ORDER", order)
        else:
            monkeypatch.delenv("EQD_ELEMENT_ORDER", raising=False)
        print(f"case {nx} {ny} {nz} {classes} {precision} order {order}", flush=True)
        s = Solver(b, sc, precision)
        info = s.layout_info()
        assert {k for k in ("tiles", "tiles_pml") if info[k] > 0} == ({tiled} if order is None else set())
        s.run(5)
        s.run(6)
        out.append({k: s.get(k) for k in KEYS})
        s.close()
    assert_same(out[0], out[1], f"{tiled} {classes} {precision}")
