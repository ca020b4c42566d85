"""FP32 PML elements in tiles form the hourglass argument u + rdampk v as the
others do: in FP64 from the differences to the element's first node, rounded
once.  Shown where that matters: a checkerboard field, whose gradients vanish
in every element of a uniform grid, with u = -float32(rdampk) v, so that
u + rdampk v is only what float32(rdampk) leaves of rdampk; formed in FP32 it
would be zero, and so would every force on a PML node."""
import numpy as np
import pytest

from eqdyna_amd import case as cases
from eqdyna_amd import mesh
from eqdyna_amd.solver import Solver


@pytest.mark.gpu
def test_hourglass_argument_is_rounded_once(monkeypatch):
    b, sc = mesh.build_case(cases.box_sw(6, 6, 3, 100.0, 3))
    b = dict(b)
    rdampk, dt = float(sc["rdampk"]), float(sc["dt"])
    r32 = float(np.float32(rdampk))
    assert abs(rdampk - r32) > 1e-9 * rdampk
    sign = 1.0 - 2.0 * (np.rint((b["meshCoor"] - b["meshCoor"][0]) / 100.0).astype(int).sum(1) % 2)
    b["velArr"] = np.repeat(sign[:, None], 3, axis=1)
    # the first step's update adds v dt to u, except on fixed nodes
    esl, eqi = b["eqNumStartIndexLoc"], b["eqNumIndexArr"]
    fixed = eqi[esl] == -1
    b["dispArr"] = -(r32 + np.where(fixed, 0.0, dt))[:, None] * b["velArr"]
    pml = (b["numOfDofPerNodeArr"] == 12) & ~fixed
    b["v1"] = b["v1"].copy()
    three = b["numOfDofPerNodeArr"] == 3
    b["v1"][eqi[esl[three][:, None] + np.arange(3)] - 1] = b["velArr"][three]
    eq = eqi[esl[pml][:, None] + np.arange(12)] - 1  # 9 split components, which the layer damps, and 3 it does not
    b["v1"][eq[:, :9]], b["v1"][eq[:, 9:]] = 0.0, b["velArr"][pml]
    monkeypatch.setenv("EQD_NO_OPERATOR_CLASSES", "1")
    force = []
    for order in ("0", "1"):
        monkeypatch.setenv("EQD_ELEMENT_ORDER", order)
        s = Solver(b, sc, "fp32")
        info = s.layout_info()
        assert info["geom_ops_pml"] == 1 and (info["tiles_pml"] > 0) == (order == "1")
        s.run(1)
        # (the value the element kernels gather: read back with its residual)
        assert np.array_equal(s.get("dispArr")[pml].astype(np.float32), -r32 * b["velArr"][pml])
        force.append(s.get("nodalForceArr")[eq[:, 9:]])
        s.close()
    size = np.max(np.abs(force[0]))
    diff = np.max(np.abs(force[1] - force[0]))
    print(f"forces on PML nodes {size:.3e}, tiles differ by {diff:.3e}", flush=True)
    # a nodal force is 8 elements' sums of some dozen rounded FP32 terms each
    assert size > 0 and diff <= 1e-5 * size
