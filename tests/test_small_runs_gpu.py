"""Lattices small enough that one block takes a whole run of steps: the same
bits as one launch a step, which a run with flux sums (LB) and a pair of equal
tracers (MP) still take.  Node counts around the edges of waves, tiles and the
rule; runs paused at odd steps, stopped by the target, by the floor of l2err,
by a negative population and by the cap."""
import numpy as np
import pytest

from laboetie_amd import lbx

PRECS = [lbx.PREC_FP64, lbx.PREC_FP32_SHIFT, lbx.PREC_FP32_STORE]


def lattice(nf):
    """nf fluid nodes at random in a box of about twice as many; 1024: four
    full tiles."""
    if nf == 1024:
        return (16, 16, 4), np.zeros(nf, np.int8)
    dims = (7, 11, -(-2 * nf // 77) + 1)
    nat = np.ones(int(np.prod(dims)), np.int8)
    nat[np.random.default_rng(nf).permutation(nat.size)[:nf]] = 0
    return dims, nat


def lb_run(L, launched, fext, target, cap, pauses):
    L.init_rest(1.0)
    L.equilibrate_begin(fext, target, max_steps=cap, flux_sums=launched)
    for t in pauses:
        r = L.equilibrate_advance(t, check=False)
        if r["status"] or r["exit_reason"]:
            break
        flow = L.flow()
    else:
        r = L.equilibrate_advance(check=False)
        flow = L.flow()
    out = [np.array([r["status"], r["steps"], r["exit_reason"]]), L.l2err_trace()]
    if r["status"] == lbx.OK:
        out += [*flow, *L.get_state()]
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("prec", PRECS)
@pytest.mark.parametrize("nf", [1, 63, 64, 65, 257, 511, 512])
def test_lb_run_in_one_block(nf, prec):
    dims, nat = lattice(nf)
    print("lb run", nf, prec, flush=True)
    fext = [1e-4, -2e-4, 3e-4]
    with lbx.Lattice(dims, nat, 0.8, precision=prec) as L:
        for what, f, target, cap, pauses, window, every in [
                ("capped", fext, 0.0, 70, (1, 2, 4, 9, 10, 41), 0, 1),
                ("target", fext, 1e-7, 4000, (5, 77), 0, 4),
                ("floor", fext, 0.0, 6000, (), 40, 1),
                ("negative", [0.9, 0.0, 0.0], 0.0, 400, (3,), 0, 1)]:
            if prec != lbx.PREC_FP64:  # FP64 measures l2err at every step and has no floor
                L.set_floor_window(window)
                L.set_check_interval(every)
            a, b = (lb_run(L, launched, f, target, cap, pauses) for launched in (False, True))
            assert len(a) == len(b), (what, a[0], b[0])
            for x, y in zip(a, b):
                assert np.array_equal(x, y, equal_nan=True), (what, a[0], b[0])


@pytest.mark.gpu
@pytest.mark.parametrize("prec", PRECS)
@pytest.mark.parametrize("form", [lbx.MP_STORED, lbx.MP_RECOMPUTED])
@pytest.mark.parametrize("ka", [0.0, 0.02])
@pytest.mark.parametrize("nf", [1, 64, 256, 257, 513, 900, 1024])
def test_mp_run_in_one_block(nf, ka, form, prec):
    dims, nat = lattice(nf)
    print("mp run", nf, ka, form, prec, flush=True)
    fext, kd, runs = [1e-4, -2e-4, 3e-4], 0.5 * ka, (1, 2, 1, 300)
    with lbx.Lattice(dims, nat, 0.8, precision=prec) as L:
        L.set_mp_coefficients(form)
        L.init_rest(1.0)
        L.equilibrate(fext, 0.0, max_steps=10)
        v1 = L.mp_init(fext, 0.01, ka, kd)
        one = [L.mp_run(n)["vacf"].reshape(n, 3) for n in runs]
        p1, d1 = L.mp_get(), L.mp_deff()
        v2 = L.mp_init_batch(fext, 0.01, [ka, ka], [kd, kd])
        two = [L.mp_run(n)["vacf"].reshape(n, 2, 3)[:, 0] for n in runs]
        assert np.array_equal(v1, v2[0])
        for a, b in zip(one, two):
            assert np.array_equal(a, b)
        for a, b in zip(p1, L.mp_get(0)):
            assert np.array_equal(a, b)
        assert np.array_equal(d1, np.asarray(L.mp_deff()).reshape(2, 3)[0])
