"""More instances in a batch than a launch grid has rows, all entering moment
propagation in the same round, and instances of very different sizes doing so."""
import numpy as np
import pytest

from laboetie_amd import lbx

pytestmark = pytest.mark.gpu

FEXT = [2e-5, -1e-5, 3e-5]


def alone(dims, nat, steps):
    with lbx.Lattice(dims, nat, 0.9) as L:
        L.init_rest(1.0)
        L.equilibrate(FEXT, 0.0, max_steps=5)
        v0 = L.mp_init(FEXT, 0.01, 0.02, 0.01)
        return np.vstack([v0, L.mp_run(steps)["vacf"]])


def test_more_instances_than_grid_rows():
    kinds = []
    for k in range(3):
        nat = np.zeros(12, np.int8)
        nat[:k] = 1
        kinds.append(((1, 3, 4), nat))
    n = 65535 + 70
    print("batch of", n, flush=True)
    want = [alone(*c, 2) for c in kinds]
    with lbx.Batch(256 * n, 12 * n, n) as B:
        for k in range(n):
            assert B.add(*kinds[k % 3], 0.9, 1.0, FEXT, 0.0, 0.01, 0.02, 0.01, 2, max_lb_steps=5) == k
        rounds = 0
        while B.round(5, 2):
            rounds += 1
            assert rounds < 9
        for k in range(n):
            assert np.array_equal(B.result(k, vacf_rows=3)["vacf"], want[k % 3]), k


def test_sizes_far_apart_enter_together():
    rng = np.random.default_rng(8)
    cases = []
    for dims in [(1, 1, 1), (100, 90, 40), (1, 40, 41), (9, 1, 1), (33, 20, 17), (1, 40, 40), (2, 3, 300), (60, 60, 60)]:
        nat = (rng.random(int(np.prod(dims))) < 0.3).astype(np.int8)
        nat[0] = 0
        cases.append((dims, nat))
    with lbx.Batch(sum(-(-int((s == 0).sum()) // 256) * 256 for _, s in cases), sum(s.size for _, s in cases),
                   len(cases)) as B:
        ids = [B.add(d, s, 0.9, 1.0, FEXT, 0.0, 0.01, 0.02, 0.01, 6, max_lb_steps=5) for d, s in cases]
        assert None not in ids
        while B.round(8, 8):
            pass
        for i, (d, s) in zip(ids, cases):
            print("sizes", d, flush=True)
            assert np.array_equal(B.result(i, vacf_rows=7)["vacf"], alone(d, s, 6))
