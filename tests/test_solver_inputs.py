"""eqd_set keeps the caller's pointers until eqd_commit has read them, so the
copies that Solver makes of inputs in another order or type must live until
then (no compute: this runs without a GPU)."""
import weakref

import numpy as np

from eqdyna_amd import solver
from fixtures import load_golden


class Lib:
    """The library's calls that Solver makes, with a look at the inputs at eqd_commit."""

    def __init__(self):
        self.copies, self.alive = [], None

    def eqd_create(self, scalars, handle):
        return 0

    def eqd_set(self, h, field, pointer, count):
        return 0

    def eqd_commit(self, h):
        self.alive = [r() is not None for r in self.copies]
        return 0

    def eqd_destroy(self, h):
        return 0


def test_converted_inputs_live_until_commit(monkeypatch):
    bundle, sc, _ = load_golden("box_sw")
    given = {k: v for k, v in bundle.items() if k in solver.INPUTS}
    given["mat"] = np.asfortranarray(given["mat"])
    given["nsmp"] = given["nsmp"].astype(np.int64)
    given["fric"] = given["fric"][:, ::-1][:, ::-1].astype(">f8")
    lib = Lib()
    convert = np.ascontiguousarray

    def watched(a, dtype=None):
        out = convert(a, dtype=dtype)
        lib.copies.append(weakref.ref(out))
        return out

    monkeypatch.setattr(solver, "lib", lambda: lib)
    monkeypatch.setattr(solver.np, "ascontiguousarray", watched)
    solver.Solver(given, sc)
    assert len(lib.copies) == len(given) and all(lib.alive)
