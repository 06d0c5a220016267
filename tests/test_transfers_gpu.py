"""Whole states and P, Pa to and from the host where the transfer buffer's
fills change: all planes of a state at once, some of them, one plane, runs of
one plane; host arrays that follow one another and that do not."""
import time

import numpy as np
import pytest

import lbref
from laboetie_amd import lbx

pytestmark = pytest.mark.gpu

# 23 planes of a state: one fill up to 11 397 box nodes, then as many planes as
# 2^18 values hold, one plane above 2^17 nodes, runs of one above 2^22 nodes
BOXES = [(1, 1, 1), (3, 5, 7), (22, 22, 22), (23, 23, 23), (50, 50, 50), (51, 51, 51), (103, 101, 101),
         (162, 162, 162)]


def medium(dims):
    rng = np.random.default_rng(int(np.prod(dims)))
    nat = (rng.random(int(np.prod(dims))) < 0.6).astype(np.int8)
    nat[-1] = 0
    return rng, nat


@pytest.mark.parametrize("prec", [lbx.PREC_FP64, lbx.PREC_FP32_SHIFT, lbx.PREC_FP32_STORE])
@pytest.mark.parametrize("dims", BOXES)
def test_state_comes_back(dims, prec):
    print("state", dims, prec, flush=True)
    rng, nat = medium(dims)
    N, fluid = nat.size, nat == 0
    rho = np.where(fluid, 1.0 + 0.05 * rng.random(N), 0.0)
    n = np.where(fluid, 0.05 + 0.01 * rng.random((19, N)), 0.0)
    j = [np.where(fluid, 0.01 * rng.random(N), 0.0) for _ in range(3)]
    junk = 7.0 * ~fluid  # a solid's values do not matter
    with lbx.Lattice(dims, nat, 0.9, precision=prec) as L:
        L.set_state((n + junk).reshape(-1), rho + junk, [a + junk for a in j])
        want = n
        if prec != lbx.PREC_FP64:  # stored as the FP32 deviation from the rest state of the first node's density
            rest = (lbx.d3q19_tables()[1] * rho[fluid][0])[:, None]
            want = np.where(fluid, rest + (n - rest).astype(np.float32).astype(np.float64), 0.0)
        for _ in range(2):
            gn, grho, gj = L.get_state()
            assert np.array_equal(gn.reshape(19, N), want)
            assert np.array_equal(grho, rho) and np.array_equal(gj, np.stack(j))
        none, grho, gj = L.get_state(populations=False)
        assert none is None and np.array_equal(grho, rho) and np.array_equal(gj, np.stack(j))


@pytest.mark.parametrize("dims", [(5, 4, 3), (35, 35, 35), (36, 36, 36), (45, 45, 45)])
def test_moments_come_back(dims):
    """P and Pa in one fill, in two, and in runs, against the restatement."""
    print("moments", dims, flush=True)
    rng, nat = medium(dims)
    fluid = nat == 0
    rho = np.where(fluid, 1.0 + 0.05 * rng.random(nat.size), 0.0)
    j = np.where(fluid, 0.01 * rng.random((3, nat.size)), 0.0)
    fext = [1e-5, 0.0, -1e-5]
    with lbx.Lattice(dims, nat, 0.9) as L:
        L.mp_init(fext, 0.01, 0.02, 0.01, flow=(rho, j))
        L.mp_run(2)
        P, Pa = L.mp_get()
    mp = lbref.MP(dims, nat, lbref.interfacial(*dims, nat), lbref.tracer_population(dims, nat, rho, j, fext), rho, 0.01,
                  0.02, 0.01)
    assert mp.run(2)[0] == 0
    assert np.array_equal(P, mp.P) and np.array_equal(Pa, mp.Pa)


def test_a_small_state_does_not_cost_a_wait_per_plane():
    """The 23 planes of a small state take little longer than its density and
    flux (5.6 times as long when each plane had a launch and a wait of its own)."""
    nat = np.zeros(64, np.int8)  # its populations are under the 16 KiB above which the runtime changes how it copies
    with lbx.Lattice((4, 4, 4), nat, 0.9) as L:
        L.init_rest(1.0)
        best = {}
        for pop in (True, False):
            t = []
            for _ in range(60):
                t0 = time.perf_counter()
                L.get_state(populations=pop)
                t.append(time.perf_counter() - t0)
            best[pop] = min(t)
    print("state / flow us", best[True] * 1e6, best[False] * 1e6, flush=True)
    assert best[True] < 3.0 * best[False]
