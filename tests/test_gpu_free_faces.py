"""Meshes without absorbing layers, whose outer nodes are all free: a tile
between two free faces owns more nodes than its workgroup updates (256), and
the rest stay with the node kernels.  Against the reference's element order:
the same bits (the tables themselves: test_tiles.py)."""
import numpy as np
import pytest

from eqdyna_amd import case as cases
from eqdyna_amd import mesh
from eqdyna_amd.solver import Solver
from test_gpu_engine import assert_same


def without_pml(b, sc):
    """The regular elements of a built case alone."""
    keep = np.flatnonzero(b["elemTypeArr"] != 2)
    used = np.unique(b["nodeElemIdRelation"][keep]) - 1
    new = np.zeros(len(b["meshCoor"]) + 1, np.int32)
    new[used + 1] = np.arange(1, len(used) + 1)
    out = dict(b)
    for k in ("meshCoor", "eqNumStartIndexLoc", "numOfDofPerNodeArr", "fnms"):
        out[k] = b[k][used]
    for k in ("elemTypeArr", "eleshp", "eledet", "elemass", "ss", "phi", "stressCompIndexArr", "eleporep", "pstrain"):
        out[k] = b[k][keep]
    out["mat"] = np.ascontiguousarray(b["mat"][:, keep])
    out["nodeElemIdRelation"] = new[b["nodeElemIdRelation"][keep]]
    out["nsmp"] = new[b["nsmp"]]
    assert np.all(out["numOfDofPerNodeArr"] == 3) and np.all(out["nsmp"] > 0)
    del out["idhist"]
    return out, dict(sc, totalNumOfNodes=len(used), totalNumOfElements=len(keep), numOfOffFaultStCount=0)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("nx,ny,nz", [(24, 11, 3), (5, 3, 30)])
def test_slab_with_free_faces(nx, ny, nz, precision, monkeypatch):
    b, sc = without_pml(*mesh.build_case(cases.box_sw(nx, nz, ny, 100.0, 3)))
    # a wave field; both nodes of a pair move together
    k = 2.0e-3 * np.array([[1.3, -0.7, 0.9], [0.8, 1.1, -1.4], [-0.6, 0.5, 1.2]])
    at = b["eqNumIndexArr"][b["eqNumStartIndexLoc"][:, None] + np.arange(3)] - 1
    b["velArr"] = 0.02 * np.cos(b["meshCoor"] @ k.T + np.arange(3))
    b["v1"] = b["v1"].copy()
    b["v1"][at] = b["velArr"]
    out = []
    for order in ("0", "1"):
        print(f"case {nx} {ny} {nz} {precision} order {order}", flush=True)
        monkeypatch.setenv("EQD_ELEMENT_ORDER", order)
        s = Solver(b, sc, precision)
        info = s.layout_info()
        assert (info["tiles"] > 0) == (order == "1")
        assert info["tile_inner_nodes"] <= 256 * info["tiles"]
        s.run(7)
        s.run(8)
        out.append({k: s.get(k) for k in ("fric", "fnft", "velArr", "dispArr", "v1", "nodalForceArr", "stressArr")})
        s.close()
    assert_same(out[1], out[0], f"slab {nx} {ny} {nz} {precision}")
    assert np.all(np.any(out[0]["velArr"] != b["velArr"], axis=1))  # every node moved
