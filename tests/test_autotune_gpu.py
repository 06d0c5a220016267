"""The autotuner leaves mp_block, which chooses nothing, as the caller set it."""
import numpy as np
import pytest

from laboetie_amd import lbx


@pytest.mark.gpu
@pytest.mark.parametrize("mp_block", [64, 128, 256])
def test_autotune_keeps_mp_block(mp_block):
    dims = (12, 11, 10)
    nat = (np.random.default_rng(1).random(1320) < 0.3).astype(np.int8)
    with lbx.Batch(2 * 1536, 2 * 1320, 2) as B:
        B.set_block(128, mp_block)
        B.add(dims, nat, 0.9, 1.0, [1e-5, 0.0, 0.0], 0.0, 0.01, 0.0, 0.0, 40, max_lb_steps=4)
        B.add(dims, nat, 0.9, 1.0, [1e-5, 0.0, 0.0], 0.0, 0.01, 0.0, 0.0, 40, max_lb_steps=40)
        for _ in range(3):
            B.round(4, 4)
        print("autotune", mp_block, flush=True)
        for _ in range(3):
            t = B.autotune(3)
            assert t["mp_block"] == mp_block and t["lb_block"] in (64, 128, 256)
            assert t["ms"]["mp64"] == t["ms"]["mp128"] == t["ms"]["mp256"] > 0
            assert all(t["ms"][k] > 0 for k in ("lb64", "lb128", "lb256", "lb_graph", "mp_graph", "mp_persistent"))
        while B.round(16, 16):
            pass
