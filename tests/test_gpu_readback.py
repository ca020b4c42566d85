"""eqd_get through the pack kernels and the pinned staging slots: a committed
state read back before any step is the given one, bit for bit (FP32 bulk mode:
its rounding), for results of less than one slot, of one and a ragged part,
and of several."""
import numpy as np
import pytest

from eqdyna_amd import case as cases
from eqdyna_amd import mesh
from eqdyna_amd.solver import Solver

SLOT = 8 << 20  # bytes of one staging slot


def scenario(nx, ny, nz, seed):
    b, sc = mesh.build_case(cases.box_sw(nx, nz, ny, 100.0, 3))
    rng = np.random.default_rng(seed)
    b = dict(b)
    b["velArr"] = rng.standard_normal(b["meshCoor"].shape)
    b["dispArr"] = rng.standard_normal(b["meshCoor"].shape)
    b["fric"] = rng.standard_normal(b["fric"].shape)
    b["fnft"] = rng.standard_normal(b["fnft"].shape)
    at = np.flatnonzero(b["numOfDofPerNodeArr"] == 3)
    eq = b["eqNumIndexArr"][b["eqNumStartIndexLoc"][at][:, None] + np.arange(3)] - 1
    b["v1"] = b["v1"].copy()
    b["v1"][eq] = b["velArr"][at]  # a 3-component node's velocity is its v1
    return b, sc


def bf16(x):
    """float32 rounded to bfloat16 (nearest even)."""
    u = x.astype(np.float32).view(np.uint32)
    u = (u + np.uint32(0x7FFF) + ((u >> np.uint32(16)) & np.uint32(1))) & np.uint32(0xFFFF0000)
    return u.view(np.float32).astype(np.float64)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("nx,ny,nz,pieces", [(4, 3, 5, 1), (69, 12, 75, 2), (69, 30, 75, 3)])
def test_readback_is_the_committed_state(nx, ny, nz, pieces, precision):
    b, sc = scenario(nx, ny, nz, seed=nx + ny)
    nn, nf = len(b["meshCoor"]), len(b["fnft"])
    assert -(-24 * nn // SLOT) == pieces and -(-800 * nf // SLOT) == min(pieces, 2)
    s = Solver(b, sc, precision)
    got = {k: s.get(k) for k in ("velArr", "dispArr", "fric", "fnft")}
    s.close()
    vel, disp = b["velArr"].copy(), b["dispArr"].copy()
    if precision == "fp32":
        free = np.ones(nn, bool)
        free[b["nsmp"].ravel() - 1] = False  # split nodes keep FP64
        hi = disp[free].astype(np.float32).astype(np.float64)
        disp[free] = hi + bf16(disp[free] - hi)
        vel[free] = vel[free].astype(np.float32)
    assert np.array_equal(got["velArr"], vel)
    assert np.array_equal(got["dispArr"], disp)
    assert np.array_equal(got["fric"], b["fric"])
    assert np.array_equal(got["fnft"], b["fnft"])


@pytest.mark.gpu
def test_no_thread_is_busy_after_a_readback():
    # the threads that empty the staging slots end with the call: what the
    # caller does next has the cores to itself
    import time
    b, sc = scenario(69, 30, 75, seed=1)
    s = Solver(b, sc, "fp32")
    time.sleep(0.5)  # (the commit's own threads come to rest)
    for k in ("velArr", "dispArr"):
        s.get(k)
    cpu = time.process_time()
    time.sleep(0.1)
    cpu = time.process_time() - cpu
    s.close()
    print(f"CPU time within 0.1 s after reading back: {cpu:.3f} s", flush=True)
    assert cpu <= 0.05  # half a core; a spinning team takes 0.7
