"""How a step is launched never changes what it computes: HIP graph replay,
every launch shape, the autotuner and batched ensembles must all reproduce
the plain eager run of each scenario bit for bit."""
import numpy as np
import pytest

from eqdyna_amd import learned
from eqdyna_amd.solver import Ensemble, Solver
from fixtures import channel_errors, channels, load_golden, undefined_slots
from test_gpu_fp32 import fp32_errors

KEYS = ["fric", "fnft", "velArr", "dispArr", "v1", "stressArr", "onFaultQuantHistSCECForm"]


def outputs(s):
    out = {k: s.get(k) for k in KEYS}
    # the per-step hypocentre record (showSourceDynamics) of every step run
    out["hypocentre"] = s.hypocentre_get(1, s.clock()[0])
    return out


def assert_same(a, b, tag):
    assert a.keys() == b.keys(), tag
    for k in a:
        x, y = a[k], b[k]
        same = np.array_equal(x, y, equal_nan=True)
        if not same:
            d = np.nanmax(np.abs(x.astype(np.float64) - y.astype(np.float64)))
            pytest.fail(f"{tag}: {k} differs (max abs {d:.3e})")


def eager_run(name, precision, chunks, guess=None):
    bundle, sc, _ = load_golden(name)
    s = Solver(bundle, sc, precision)
    s.set_graph(False)  # every step launched (no replay even for long runs)
    if guess is not None:
        s.set_guess(*guess)
    for n in chunks:
        s.run(n)
    out = outputs(s)
    s.close()
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("name,precision", [("box_rsf4", "fp64"), ("box_sw", "fp32"), ("box_q", "fp64")])
def test_graph_replay_matches_eager(name, precision):
    print(f"case {name} {precision}", flush=True)
    bundle, sc, _ = load_golden(name)
    nstep = int(sc["nstep"])
    chunks = [1, 7, nstep - 8 - 5, 5]
    ref = Solver(bundle, sc, precision)
    ref.set_graph(False)
    s = Solver(bundle, sc, precision)
    s.set_graph(True)
    done = 0
    for n in chunks:
        # every call replays the captured step n times, then synchronizes; the
        # eager run of the same chunk goes in between, and each chunk's state
        # is compared, so every replay of the graph is checked
        s.run(n)
        ref.run(n)
        done += n
        assert s.clock()[0] == ref.clock()[0] == done
        assert_same(outputs(s), outputs(ref), f"{name} graph after {done} steps")
    s.close()
    ref.close()


@pytest.mark.gpu
@pytest.mark.parametrize("name,precision", [("box_rsf4", "fp64"), ("box_q", "fp32"), ("box_tp", "fp64")])
def test_step_start_in_element_launch_matches_own_launch(name, precision, monkeypatch):
    # the clock advance and the off-fault stations carried by the first
    # blocks of the regular-element launch (default) and launched on their
    # own (EQD_STEP_START_LAUNCH=1): the same clock, station rows and state,
    # over runs split so that the last-step flag is set more than once
    res = []
    for own in ("0", "1"):
        monkeypatch.setenv("EQD_STEP_START_LAUNCH", own)
        bundle, sc, _ = load_golden(name)
        s = Solver(bundle, sc, precision)
        n = int(sc["nstep"])
        s.run(n // 3)
        s.run(n - n // 3)
        assert s.clock()[0] == n
        res.append(dict(outputs(s), stations=s.get("OffFaultStGramSCEC")))
        s.close()
    assert_same(res[0], res[1], f"{name} {precision} step start in the element launch vs its own launch")
    assert np.any(res[0]["stations"] != 0) and np.array_equal(res[0]["stations"], res[1]["stations"])


@pytest.mark.gpu
@pytest.mark.parametrize("name,precision", [("box_rsf4", "fp64"), ("box_dip", "fp64"), ("box_rough", "fp32"),
                                            ("box_q", "fp32")])
def test_slot_major_node_gather_matches_csr(name, precision, monkeypatch):
    # the free nodes' gather from the slot-major table (default) and from the
    # CSR table (EQD_NODE_ELL=0) add the same forces in the same order
    res = []
    for ell in ("1", "0"):
        monkeypatch.setenv("EQD_NODE_ELL", ell)
        bundle, sc, _ = load_golden(name)
        s = Solver(bundle, sc, precision)
        s.run(int(sc["nstep"]))
        res.append(outputs(s))
        s.close()
    assert_same(res[0], res[1], f"{name} {precision} slot-major vs CSR gather")


@pytest.mark.gpu
def test_sampled_timing_counts_and_keeps_results():
    # per-kernel events on every 4th step of a run: the timers count exactly
    # those launches, and timing never changes what the steps compute
    bundle, sc, _ = load_golden("box_rsf4")
    n = int(sc["nstep"])
    s = Solver(bundle, sc)
    s.set_timing(4)
    s.run(n)
    for k in ("element", "element_pml", "node", "node_pml", "fault"):
        ms, launches = s.kernel_time(k)
        assert launches == (n + 3) // 4 and ms > 0, (k, ms, launches)
    timed = outputs(s)
    s.close()
    s = Solver(bundle, sc)
    s.run(n)
    assert_same(outputs(s), timed, "sampled timing")
    s.close()


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["box_rsf4", "box_layered"])
def test_launch_shapes_do_not_change_results(name):
    print(f"case {name}", flush=True)
    bundle, sc, _ = load_golden(name)
    nstep = int(sc["nstep"])
    ref = eager_run(name, "fp64", [nstep])
    for block, remap in ((64, 1), (128, 0), (256, 1)):
        s = Solver(bundle, sc, "fp64")
        for kind in ("element", "element_pml", "node", "node_pml"):
            s.set_launch(kind, block, remap)
        s.set_launch("fault", 64 if block == 64 else 128, 0)
        s.run(nstep)
        assert_same(outputs(s), ref, f"{name} block {block} remap {remap}")
        s.close()


@pytest.mark.gpu
def test_tuner_restores_state_and_keeps_results():
    name = "box_rsf3"
    bundle, sc, _ = load_golden(name)
    nstep = int(sc["nstep"])
    ref = eager_run(name, "fp64", [10, nstep - 10])
    s = Solver(bundle, sc, "fp64")
    s.run(10)
    before = outputs(s)
    rep = s.tune(steps=3)
    print(f"tuner report: {rep}", flush=True)
    assert set(rep) == {"element", "element_pml", "node", "node_pml", "fault"}
    for k, v in rep.items():
        assert v["ms"] > 0 and len(v["candidates"]) == (2 if k == "fault" else 6)
        assert (v["block"], v["remap"]) == s.get_launch()[k]
    assert s.clock()[0] == 10
    assert_same(outputs(s), before, "state after tuning")
    s.run(nstep - 10)
    assert_same(outputs(s), ref, "run after tuning")
    s.close()


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_ensemble_matches_individual_runs(precision):
    # scenarios of different sizes and physics: slip and time weakening, both
    # rate-and-state laws (two with the learned guess), Q, a rough fault, and
    # two scenarios drawn like the c5 ensemble's (layered medium, von Karman
    # tau_0, drawn hypocentre)
    names = ["box_sw", "box_tw", "box_rsf3", "box_rsf4", "box_q", "box_rough", "box_layered", "box_c5sw",
             "box_c5rsf"]
    params, _ = learned.load()
    guesses = {"box_rsf4": (params, 6, 0.5), "box_rsf3": (None, 4, 0.5), "box_c5rsf": (params, 6, 0.5)}
    steps = {}
    refs = {}
    for n in names:
        _, sc, _ = load_golden(n)
        steps[n] = int(sc["nstep"])
        print(f"individual {n} {precision}", flush=True)
        refs[n] = eager_run(n, precision, [steps[n]], guesses.get(n))
    common = min(steps.values())
    members = []
    for n in names:
        bundle, sc, _ = load_golden(n)
        s = Solver(bundle, sc, precision)
        if n in guesses:
            s.set_guess(*guesses[n])
        members.append(s)
    ens = Ensemble(members)
    print(f"ensemble of {len(members)} scenarios, {common} common steps", flush=True)
    ens.run(3)
    ens.run(common - 3)
    ens.close()
    for n, s in zip(names, members):
        assert s.clock()[0] == common
        if steps[n] > common:
            s.run(steps[n] - common)  # back on its own engine after the ensemble
        assert_same(outputs(s), refs[n], f"ensemble member {n}")
        # and each member against the reference's own FP64 run of its inputs:
        # the error bars of the faster modes for every member, the FP64 bar
        # (1e-9 per channel) for the plain FP64 members; box_rough's reference
        # run moves by about 1e-7 under a one-ulp input change, so it is held
        # to the conditioning bar of test_gpu_parity (at most 1e-6)
        out = s.outputs()
        s.close()
        _, sc, fix = load_golden(n)
        e = fp32_errors(out, fix, sc["dt"])
        skip = undefined_slots(sc)
        ch = channel_errors(channels(out, skip), channels(fix, skip))
        worst = max(ch, key=ch.get)
        print(f"ensemble member {n} ({precision}{', guess' if n in guesses else ''}) vs reference: {e}; "
              f"worst channel {worst} {ch[worst]:.2e}", flush=True)
        assert e["rupture_flips"] == 0 and e["rupture_time_mean_dt"] <= 0.5 and e["peak_slip_rate_rel"] <= 0.01
        if precision == "fp64" and n not in guesses:
            assert ch[worst] <= (1e-6 if n == "box_rough" else 1e-9), (n, worst, ch[worst])


@pytest.mark.gpu
def test_ensemble_tuner():
    names = ["box_sw", "box_rsf4", "box_layered"]
    members = []
    for n in names:
        bundle, sc, _ = load_golden(n)
        members.append(Solver(bundle, sc, "fp32"))
    ens = Ensemble(members)
    rep = ens.tune(steps=2)
    print(f"ensemble tuner report: {rep}", flush=True)
    assert "element" in rep and "fault" in rep
    assert all(m.clock()[0] == 0 for m in members)
    ens.run(20)
    ens.close()
    for m in members:
        assert m.clock()[0] == 20
        m.close()


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["box_rsf4", "box_dip", "box_rough", "box_tp"])
def test_element_order_does_not_change_results(name, monkeypatch):
    # elements in bricks (EQD_ELEMENT_ORDER=1) or in reference order: every
    # node still sums its elements in ascending reference id
    print(f"case {name}", flush=True)
    bundle, sc, _ = load_golden(name)
    nstep = int(sc["nstep"])
    monkeypatch.setenv("EQD_ELEMENT_ORDER", "0")
    ref = eager_run(name, "fp64", [nstep])
    monkeypatch.setenv("EQD_ELEMENT_ORDER", "1")
    got = eager_run(name, "fp64", [nstep])
    assert_same(got, ref, f"{name} brick order")


@pytest.mark.gpu
@pytest.mark.parametrize("name,precision", [("box_sw", "fp64"), ("box_rsf4", "fp32"), ("box_q", "fp32"),
                                            ("box_plastic", "fp64"), ("box_dip", "fp64"), ("box_rough", "fp32"),
                                            ("box_tp", "fp64"), ("box_hg2", "fp64")])
def test_merged_launches_match_launches_apart(name, precision, monkeypatch):
    # both element classes in one launch, fault pairs and nodes in another
    # (the default for small scenarios), against one launch per kind on two
    # streams: every launch does the same work per element, node and pair; with
    # timer events on every third step both forms alternate within a run
    bundle, sc, _ = load_golden(name)
    n = int(sc["nstep"])
    guess = (learned.load()[0], 6, 0.5) if name in ("box_rsf4", "box_rough") else None
    res = []
    for merge, timing in (("0", 0), ("1", 0), ("1", 3)):
        print(f"case {name} {precision} merge {merge} timing {timing}", flush=True)
        monkeypatch.setenv("EQD_MERGE", merge)
        s = Solver(bundle, sc, precision)
        if guess:
            s.set_guess(*guess)
        s.set_timing(timing)
        s.run(n // 3)
        s.run(n - n // 3)
        res.append(dict(outputs(s), stations=s.get("OffFaultStGramSCEC")))
        s.close()
    assert_same(res[1], res[0], f"{name} {precision} merged")
    assert_same(res[2], res[0], f"{name} {precision} merged, sampled timing")


@pytest.mark.gpu
def test_merged_ensemble_replay(monkeypatch):
    # slip weakening alone shares one kernel variant of each kind
    names = ["box_sw", "box_c5sw", "box_layered"]
    out = {}
    for merge in ("0", "1"):
        monkeypatch.setenv("EQD_MERGE", merge)
        members = [Solver(*load_golden(n)[:2], "fp32") for n in names]
        e = Ensemble(members)
        for _ in range(3):  # replays of the captured step
            e.run(6)
        out[merge] = [outputs(m) for m in members]
        e.close()
        for m in members:
            m.close()
    for n, a, b in zip(names, out["1"], out["0"]):
        assert_same(a, b, f"member {n} merged")


@pytest.mark.gpu
def test_launch_shape_of_elements_in_tiles(monkeypatch):
    # a tile is a workgroup of 256 whatever block size is asked for, and that is
    # what is reported and tried; the node kinds take any
    bundle, sc, _ = load_golden("box_rsf4")
    n = 12
    out = []
    for order in ("0", "1"):
        monkeypatch.setenv("EQD_ELEMENT_ORDER", order)
        s = Solver(bundle, sc)
        for kind in ("element", "element_pml", "node"):
            s.set_launch(kind, 64, 1)
        got = s.get_launch()
        block = 64 if order == "0" else 256
        assert got["element"] == (block, 1) and got["element_pml"] == (block, 1) and got["node"] == (64, 1)
        s.run(n)
        rep = s.tune(2)
        for kind in ("element", "element_pml"):
            shapes = [tuple(c[:2]) for c in rep[kind]["candidates"]]
            assert shapes == [(b, r) for b in ((64, 128, 256) if order == "0" else (256,)) for r in (0, 1)]
            assert (rep[kind]["block"], rep[kind]["remap"]) == s.get_launch()[kind]
        s.run(n)
        out.append(outputs(s))
        s.close()
    assert_same(out[1], out[0], "tiles with launch shapes set and tuned")


@pytest.mark.gpu
@pytest.mark.parametrize("ensemble", [False, True])
def test_tuner_weighs_shared_launches(ensemble, monkeypatch):
    # a small scenario runs two launches a step unless it is told otherwise
    # (about half the time of one launch per kind): tuning keeps that, a launch
    # shape set by the caller and EQD_MERGE=0 do not, and the results are the same
    bundle, sc, _ = load_golden("box_sw")
    n = 40
    ref = eager_run("box_sw", "fp64", [n])
    for merge in ("", "0"):
        if merge:
            monkeypatch.setenv("EQD_MERGE", merge)
        members = [Solver(bundle, sc) for _ in range(2 if ensemble else 1)]
        top = Ensemble(members) if ensemble else members[0]
        rep = top.tune(4)
        print(f"merge '{merge}' ensemble {ensemble}: {rep}", flush=True)
        assert all(v["merged"] == (merge == "") for v in rep.values())
        top.run(n // 2)
        if not ensemble:
            top.set_launch("node", 128, 0)
        top.run(n - n // 2)
        if ensemble:
            top.close()
        for s in members:
            assert_same(outputs(s), ref, f"tuned, merge '{merge}'")
            s.close()
