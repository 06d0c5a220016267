"""lbx_footprint_bytes bounds what a context allocates."""
import ctypes

import numpy as np
import pytest

from laboetie_amd import lbx

PRECS = [lbx.PREC_FP64, lbx.PREC_FP32_SHIFT, lbx.PREC_FP32_STORE]


@pytest.mark.parametrize("prec", PRECS)
@pytest.mark.parametrize("dims", [(48, 48, 48), (128, 128, 128), (256, 256, 256), (1, 512, 512)])
def test_footprint_counts_the_stored_probabilities(dims, prec):
    """A box of fluid in full tiles: per node of a propagation the 18
    probabilities, rem, u*, P and Pa twice per tracer, the slot table and the
    node; per tile its halo list."""
    N, pop = int(np.prod(dims)), 8 if prec == lbx.PREC_FP64 else 4
    for ntr in (1, 3, 4):
        got = lbx.footprint_bytes(*dims, prec, ntr) - lbx.footprint_bytes(*dims, prec, 0)
        assert got >= N * (18 * pop + 8 + 3 * pop + 24 + 4 + 96 * ntr) + N / 256 * 344 * 4


@pytest.mark.gpu
@pytest.mark.parametrize("prec", PRECS)
@pytest.mark.parametrize("what", ["open", "noise", "channels"])
def test_footprint_bounds_the_memory_in_use(what, prec):
    dims = (128, 128, 128)
    if what == "open":
        nat = np.zeros(128 ** 3, np.int8)
    elif what == "noise":  # bricks that hold a little more than half a tile: the most entries per node
        nat = (np.random.default_rng(1).random(128 ** 3) >= 0.55).astype(np.int8)
    else:
        x = np.arange(128) % 8 >= 5
        nat = np.broadcast_to(x[:, None] | x[None, :], dims).astype(np.int8).reshape(-1)

    def free():  # the HIP runtime that the library is linked to
        left, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert lbx.lib().hipMemGetInfo(ctypes.byref(left), ctypes.byref(total)) == 0
        return left.value

    with lbx.Lattice((4, 4, 4), np.zeros(64, np.int8), 0.9, precision=prec) as L:  # the runtime's own memory
        L.init_rest(1.0)
        L.mp_init([1e-5, 0.0, 0.0], 0.01, 0.02, 0.01)
        L.mp_run(2)
    for ntr in (1, 3):
        for form in (lbx.MP_AUTO, lbx.MP_STORED):
            print("footprint", what, prec, ntr, form, flush=True)
            before = free()
            with lbx.Lattice(dims, nat, 0.9, precision=prec) as L:
                L.set_mp_coefficients(form)
                L.init_rest(1.0)
                L.equilibrate([1e-5, 0.0, 0.0], 0.0, max_steps=4)
                L.mp_init_batch([1e-5, 0.0, 0.0], 0.01, [0.02] * ntr, [0.01] * ntr)
                L.mp_run(2)
                L.get_state(populations=False)
                used = before - free()
            bound = lbx.footprint_bytes(*dims, prec, ntr)
            print(used, bound, flush=True)
            assert used <= bound + (16 << 20)  # allocations are rounded to the driver's pages


def test_footprint_beyond_32_bit_counts():
    """The sizes are 64-bit numbers, also of boxes and batches that are refused."""
    for prec in PRECS:
        for ntr in (0, 1, 3):
            small, large = (lbx.footprint_bytes(n, n, n, prec, ntr) for n in (800, 3200))
            assert 60 < large / small < 68, (prec, ntr, small, large)
        small, large = (lbx.Batch.footprint_bytes(n, n, 1, prec) for n in (1 << 27, 1 << 41))
        assert 1.6e4 < large / small < 1.7e4, (prec, small, large)
