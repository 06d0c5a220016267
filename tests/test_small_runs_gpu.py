"""Lattices small enough that one block takes a whole chunk of MP steps: the
same bits as one launch a step, which a pair of equal tracers still takes.
Node counts around the edges of waves, tiles and the rule."""
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
