"""Every way in which a run of steps by one block ends (lattices of up to 512
nodes): the target, the l2err floor of the FP32 forms, a negative population, the
cap.  Status, step, reason, l2err record and state against the restatement; the
exit is stated with each case, so that each one is known to be taken."""
import numpy as np
import pytest

import lbref
from test_small_runs_gpu import lattice

from laboetie_amd import lbx

NAMES = {lbx.PREC_FP64: "fp64", lbx.PREC_FP32_SHIFT: "shift", lbx.PREC_FP32_STORE: "store"}
FEXT = [1e-4, -2e-4, 3e-4]
LATTICES = {"slit64": ((4, 4, 6), None), "slit256": ((4, 4, 18), None), "slit512": ((4, 4, 34), None),
            "random257": lattice(257), "random511": lattice(511), "random512": lattice(512)}
ALL = "fp64 shift store"
# (lattice, fext, target, cap, floor window, steps between checks in stage 2, forms, exit)
CASES = [(name, FEXT, 0.0, 70, 0, 1, ALL, "cap") for name in LATTICES]
CASES += [(name, [0.9, 0.0, 0.0], 0.0, 400, 0, 1, ALL, "negative") for name in LATTICES]
CASES += [(name, FEXT, 1e-7, 4000, 0, 4, ALL, "converged") for name in ("slit64", "slit256")]
CASES += [(name, FEXT, 1e-7, 4000, 0, 4, "shift store", "converged") for name in ("random257", "random511", "random512")]
CASES += [(name, FEXT, 0.0, 6000, 40, 1, "shift store", "floor") for name in ("slit64", "slit256")]
CASES += [("slit512", FEXT, 0.0, 6000, 40, 1, "shift", "floor")]
WANT = {"cap": (lbx.OK, lbx.EXIT_CAP), "converged": (lbx.OK, lbx.EXIT_CONVERGED), "floor": (lbx.OK, lbx.EXIT_FLOOR),
        "negative": (lbx.ERR_NEG_POP, 0)}


@pytest.mark.gpu
@pytest.mark.parametrize("prec", NAMES)
@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}-{c[7]}")
def test_run_ends(case, prec):
    name, fext, target, cap, window, every, forms, end = case
    if NAMES[prec] not in forms:
        return
    print("run exit", name, end, NAMES[prec], flush=True)
    dims, nat = LATTICES[name]
    if nat is None:
        nat = lbx.build_geometry(1, *dims)
    if prec == lbx.PREC_FP64:
        ref = lbref.equilibrate(dims, nat, 0.8, 1.0, fext, target, max_steps=cap)
    else:
        ref = lbref.equilibrate_shift(dims, nat, 0.8, 1.0, fext, target, max_steps=cap, floor_window=window,
                                      arith="fp32" if prec == lbx.PREC_FP32_SHIFT else "fp64", check_every=every)
    assert (int((nat == 0).sum()) <= 512 and ref["exit_reason"] == WANT[end][1]
            and (ref["status"] != 0) == (WANT[end][0] != 0))
    with lbx.Lattice(dims, nat, 0.8, precision=prec) as L:
        if prec != lbx.PREC_FP64:
            L.set_floor_window(window)
            L.set_check_interval(every)
        L.init_rest(1.0)
        r = L.equilibrate(fext, target, max_steps=cap, check=False)
        assert (r["status"], r["exit_reason"]) == WANT[end]
        assert r["steps"] == ref["steps"]
        measured = r["steps"] - (r["status"] != lbx.OK)  # the step that finds a negative population has none
        assert np.array_equal(r["l2err"], ref["l2err"][:measured], equal_nan=True)
        if r["status"] == lbx.OK:
            n, rho, j = L.get_state()
            assert np.array_equal(n, ref["n"]) and np.array_equal(rho, ref["rho"]) and np.array_equal(j, ref["j"])
