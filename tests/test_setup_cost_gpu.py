"""What setting up again costs: a program that propagates one set of tracers
after another on a context pays for the set-up's kernels, not for the arrays."""
import time

import numpy as np
import pytest

from laboetie_amd import lbx

pytestmark = pytest.mark.gpu


def again_us(n, **kw):
    nat = (np.random.default_rng(n).random(n ** 3) >= 0.6).astype(np.int8)
    nat[0] = 0
    with lbx.Lattice((n, n, n), nat, 0.9, **kw) as L:
        L.init_rest(1.0)
        L.mp_init([1e-6, 0.0, 0.0], 0.01, 0.01, 0.01)
        t = []
        for _ in range(15):
            t0 = time.perf_counter()
            L.mp_init([1e-6, 0.0, 0.0], 0.01, 0.01, 0.01)
            t.append(time.perf_counter() - t0)
    return sorted(t)[7] * 1e6


@pytest.mark.parametrize("prec", [lbx.PREC_FP64, lbx.PREC_FP32_SHIFT])
def test_propagating_again_takes_no_new_arrays(prec):
    """64^3 nodes against 24^3: 20 times the nodes, but on this card still a
    launch's time (a set-up that allocated each array again: 33 times as long)."""
    small, large = again_us(24, precision=prec), again_us(64, precision=prec)
    print("mp_init again us", small, large, flush=True)
    assert large < 12.0 * small


@pytest.mark.parametrize("prec", [lbx.PREC_FP64, lbx.PREC_FP32_SHIFT])
def test_one_context_through_many_propagations(prec):
    """More and fewer tracers, with and without adsorption, and both stored
    forms on one context: each propagation as on a context of its own."""
    dims = (23, 19, 17)
    nat = (np.random.default_rng(3).random(int(np.prod(dims))) >= 0.7).astype(np.int8)
    nat[0] = 0
    fext = [1e-5, -2e-5, 0.0]
    runs = [(1, 0.02, lbx.MP_AUTO), (4, 0.02, lbx.MP_RECOMPUTED), (1, 0.0, lbx.MP_STORED), (3, 0.0, lbx.MP_STORED),
            (4, 0.03, lbx.MP_STORED), (2, 0.01, lbx.MP_AUTO)]

    def propagate(L, ntr, ka, form):
        L.set_mp_coefficients(form)
        v0 = L.mp_init_batch(fext, 0.01, [ka * (t + 1) for t in range(ntr)], [0.01 if ka else 0.0] * ntr)
        return [v0, L.mp_run(7)["vacf"], L.mp_deff()] + [a for t in range(ntr) for a in L.mp_get(t)]

    def fresh():
        L = lbx.Lattice(dims, nat, 0.9, precision=prec)
        L.init_rest(1.0)
        L.equilibrate(fext, 0.0, max_steps=12)
        return L

    with fresh() as one:
        for r in runs + runs[::-1]:
            print("propagate", prec, r, flush=True)
            got = propagate(one, *r)
            with fresh() as own:
                for a, b in zip(got, propagate(own, *r)):
                    assert np.array_equal(a, b)
