"""Elements in tiles, whose inner nodes the element kernels sum and update
themselves (the default from 163,840 regular and 196,608 PML elements on,
EQD_ELEMENT_ORDER=1 on any mesh), against the reference's element order: a
node sums the same forces in the same order, so every output is the same bit
for bit."""
import numpy as np
import pytest

from eqdyna_amd.solver import Ensemble, Solver
from fixtures import channel_errors, channels, load_golden
from test_gpu_engine import assert_same, outputs


def solver(name, precision, tiles, monkeypatch):
    monkeypatch.setenv("EQD_ELEMENT_ORDER", "1" if tiles else "0")
    bundle, sc, _ = load_golden(name)
    s = Solver(bundle, sc, precision)
    info = s.layout_info()
    for k in ("tiles", "tile_inner_nodes", "tiles_pml", "tile_inner_nodes_pml"):
        assert (info[k] > 0) == tiles, k
    return s, bundle, sc


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["box_sw", "box_q", "box_plastic", "box_hg2", "box_layered", "box_dip", "box_rough",
                                  "box_c5rsf"])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_tiles_match_reference_order(name, precision, monkeypatch):
    if name == "box_plastic" and precision == "fp32":
        pytest.skip("the FP32 mode is not meant for lithostatic stresses")
    # operators from class tables and from memory; runs split so that the
    # stored F/m of the last step is applied by the next run; records of all
    # nodes at the step they belong to; station rows
    res = []
    for tiles, classes in ((False, "0"), (True, "0"), (False, "1"), (True, "1")):
        monkeypatch.setenv("EQD_NO_OPERATOR_CLASSES", classes)
        monkeypatch.setenv("EQD_GEOM_OPS", "0")  # operators rebuilt in the kernels: test_modal_operators
        print(f"case {name} {precision} tiles {tiles} per-element operators {classes}", flush=True)
        s, bundle, sc = solver(name, precision, tiles, monkeypatch)
        n = int(sc["nstep"])
        s.record(np.arange(1, len(bundle["meshCoor"]) + 1, dtype=np.int32), 3, n)
        s.run(n // 3)
        s.run(n - n // 3)
        vel, rate = s.record_get(n)
        o = dict(outputs(s), stations=s.get("OffFaultStGramSCEC"), force=s.get("nodalForceArr"), vel=vel, rate=rate)
        assert vel.shape[0] == (n - 1) // 3 + 1 and np.any(vel != 0)
        res.append(o)
        s.close()
    assert_same(res[1], res[0], f"{name} {precision} tiles")
    assert_same(res[3], res[2], f"{name} {precision} tiles, per-element operators")


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["box_rough", "box_q", "box_hg2", "box_plastic", "box_tw"])
def test_modal_operators(name, monkeypatch):
    # FP32, operators rebuilt from corner coordinates: tiles form them per mode
    # (split8, join8), the reference's order node by node.  The two round
    # differently; both have FP32's bars against the FP64 run: rupture times
    # within half a step, and every channel within 1e-4 of the other (about a
    # thousand roundings of 6e-8 that add up over the run)
    monkeypatch.setenv("EQD_NO_OPERATOR_CLASSES", "1")
    out = {}
    for tiles in (False, True):
        print(f"case {name} tiles {tiles}", flush=True)
        s, bundle, sc = solver(name, "fp32", tiles, monkeypatch)
        assert s.layout_info()["geom_ops_regular"] == 1
        s.run(int(sc["nstep"]))
        out[tiles] = s.outputs()
        s.close()
    d = channel_errors(channels(out[True]), channels(out[False]))
    worst = max(d, key=d.get)
    print(f"[{name}] modal against node by node: worst channel {worst} {d[worst]:.2e}", flush=True)
    assert d[worst] <= 1e-4
    assert np.max(np.abs(out[True]["fnft"] - out[False]["fnft"])) <= 0.5 * float(sc["dt"])


@pytest.mark.gpu
def test_ensemble_of_scenarios_with_and_without_tiles(monkeypatch):
    names = ["box_c5sw", "box_sw", "box_c5rsf", "box_layered"]
    want, members = [], []
    for n in names:
        s, _, _ = solver(n, "fp32", False, monkeypatch)
        s.run(20)
        want.append(outputs(s))
        s.close()
    for i, n in enumerate(names):
        members.append(solver(n, "fp32", i % 2 == 1, monkeypatch)[0])
    e = Ensemble(members)
    for k in range(4):  # replays of the captured step, each chunk ending in a stored F/m
        e.run(5)
    for n, m, w in zip(names, members, want):
        assert_same(outputs(m), w, f"member {n}")
    e.close()
    for m in members:
        m.close()


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_nan_in_a_tile_is_named_by_the_reference_order(precision, monkeypatch):
    # three free nodes poisoned, the highest first: tiles store nodes in
    # another order, the report names the lowest id of the reference
    from eqdyna_amd.solver import EqdError
    bundle, sc, _ = load_golden("box_sw")
    split = set(int(x) for x in bundle["nsmp"].ravel())
    three = [i for i in np.flatnonzero(bundle["numOfDofPerNodeArr"] == 3) + 1 if int(i) not in split]
    b = dict(bundle, v1=bundle["v1"].copy())
    for i in (three[-5], three[len(three) // 2], three[len(three) // 3]):
        b["v1"][bundle["eqNumIndexArr"][bundle["eqNumStartIndexLoc"][i - 1]] - 1] = np.nan
    got = []
    for order in ("0", "1"):
        monkeypatch.setenv("EQD_ELEMENT_ORDER", order)
        s = Solver(b, sc, precision)
        with pytest.raises(EqdError):
            s.run(3)
        got.append((s.nan_info(), s.clock()))
        s.close()
    assert got[0] == got[1]
