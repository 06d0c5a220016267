"""The tiles of moment propagation (lbx_mp.h) with the bricks that a box is cut
into: whole and merged bricks, tiles cut once and several times because their
halo outgrows a brick's, and a lattice that runs out of tiles on the way and
takes the general step, some of whose neighbours have no LDS slot; lattices whose
bricks fill little over half a tile, with halves of them.  P, Pa bit for bit
against the restatement, in the FP32 forms each of several tracers also as alone;
batch instances: VACF and D_eff are the single lattice's bits.

layout() restates the cut and the grouping, so that each case is known to be
the kind it is meant to be."""
import sys

import numpy as np
import pytest

import lbref
from test_mp_tiles_gpu import C, noise, pockets, run_single

from laboetie_amd import lbx

HALO, SLOTS = 344, 766  # halo nodes of a brick, of a general tile


def brick(lx, ly, lz):
    """8 nodes along x; y and z of the least shell per node, the first of equals."""
    bx, best = min(lx, 8), None
    for y in range(1, min(ly, 256 // bx) + 1):
        z = min(lz, 256 // (bx * y))
        outer, vol = min(bx + 2, lx) * min(y + 2, ly) * min(z + 2, lz), bx * y * z
        if outer - vol <= HALO and (best is None or (outer + 40) / vol < best[0]):
            best = ((outer + 40) / vol, y, z)
    return bx, best[1], best[2]


def settle(fluid, b, inner, bound):
    """(tiles, times that the worst one is cut, largest halo of the uncut ones)
    with bricks b, `inner` of them along z walked together; no tiles: it takes
    more than `bound`."""
    lz, ly, lx = fluid.shape
    nb = [-(-n // k) for n, k in zip((lx, ly, lz), b)]
    cx, cy = min(8, nb[0]), min(8, nb[1])
    walk = [(x0 + x, y0 + y, z0 + z) for y0 in range(0, nb[1], cy) for x0 in range(0, nb[0], cx)
            for z0 in range(0, nb[2], inner) for y in range(cy) for x in range(cx) for z in range(inner)]
    nodes = [np.argwhere(fluid[z * b[2]:(z + 1) * b[2], y * b[1]:(y + 1) * b[1], x * b[0]:(x + 1) * b[0]])
             + (z * b[2], y * b[1], x * b[0]) for x, y, z in walk]

    def group(run):
        tiles = []
        for o in range(0, len(walk), run):
            fresh = True
            for n in nodes[o:o + run]:
                if len(n) == 0:
                    continue
                if fresh or sum(map(len, tiles[-1])) + len(n) > 256:
                    tiles.append([])
                fresh = False
                tiles[-1].append(n)
        return tiles

    def halo(t):
        own = {tuple(v) for n in t for v in n}
        return sum(bool(fluid[v]) for v in {((z + c[2]) % lz, (y + c[1]) % ly, (x + c[0]) % lx)
                                            for z, y, x in own for c in C} - own)

    def parts(t, level):
        out, at = {}, 0
        for n in t:
            out.setdefault((at << level) >> 8, []).append(n)
            at += len(n)
        return list(out.values())

    tiles = group(128 * inner)
    if len(tiles) > bound and inner == 1:
        tiles = group(len(walk))
    halos = list(map(halo, tiles))
    if len(tiles) > bound:
        return 0, 0, max(halos)
    todo, level = [t for t, h in zip(tiles, halos) if h > HALO], 0
    kept = total = len(tiles) - len(todo)
    total += len(todo)
    while todo:
        level += 1
        cut = [parts(t, level) for t in todo]
        total = kept + sum(map(len, cut))
        if total > bound:
            return 0, level, max(halos)
        fits = [max(map(halo, p)) <= HALO for p in cut]
        kept += sum(len(p) for p, f in zip(cut, fits) if f)
        todo = [t for t, f in zip(todo, fits) if not f]
    return total, level, max(halos)


def layout(dims, nat):
    """(times that the worst tile is cut, or "general", or "halves" / "whole" for
    a lattice that tries halves of its bricks and takes them or not; largest
    halo of the uncut tiles)"""
    lx, ly, lz = dims
    fluid, b = nat.reshape(lz, ly, lx) == 0, brick(*dims)
    nf = int(fluid.sum())
    whole = settle(fluid, b, 1, 2 * -(-nf // 256))
    if not whole[0]:
        return "general", whole[2]
    if whole[0] >= 256 and whole[0] * 179 > nf and b[2] > 1:
        half = settle(fluid, (b[0], b[1], -(-b[2] // 2)), 2, whole[0] - whole[0] // 10)
        return ("halves", half[2]) if half[0] else ("whole", whole[2])
    return whole[1], whole[2]


def channels(dims, w, period):
    """Square channels w wide along z."""
    lx, ly, lz = dims
    x, y = np.arange(lx) % period >= w, np.arange(ly) % period >= w
    return np.broadcast_to(y[:, None] | x[None, :], (lz, ly, lx)).astype(np.int8).reshape(-1)


def corner_lines():
    """Channels 2 by 2 wide along z on the edges where four columns of bricks
    meet: each column holds a line of every channel, and all neighbours of a
    line but its own are other columns'."""
    dims = (128, 64, 128)
    at = np.meshgrid([0, 63, 64, 127], [0, 31, 32, 63], np.arange(128), indexing="ij")
    return dims, pockets(dims, [v.ravel() for v in at])


def box(*dims):
    return dims, np.zeros(int(np.prod(dims)), np.int8)


CASES = {
    "whole_bricks": (*box(16, 8, 16), 0),
    "merged": (*noise((48, 48, 32), 0.85, 2), 0),
    "flat": (*noise((1, 60, 70), 0.4, 4), 0),
    "channels": ((64, 64, 16), channels((64, 64, 16), 5, 8), 1),
    "ragged_box": (*box(33, 33, 33), 3),
    "ragged_noise": (*noise((37, 21, 11), 0.3, 1), 2),
    "fine_noise": (*noise((64, 64, 64), 0.42, 6), "halves"),
    "fine_ragged": (*noise((61, 67, 50), 0.45, 7), "halves"),
    "wide_channels": ((64, 64, 48), channels((64, 64, 48), 7, 9), "whole"),
    "corner_lines": (*corner_lines(), "general"),
}
FEXT, KA, KD = [2e-5, -1e-5, 3e-5], [0.02, 0.0, 0.05], [0.01, 0.0, 0.01]


def test_cases_are_of_their_kinds():
    beyond = False
    for name, (dims, nat, want) in CASES.items():
        kind, halo = layout(dims, nat)
        print(name, brick(*dims), kind, halo)
        assert kind == want, (name, kind, halo)
        beyond = beyond or (kind == "general" and halo > SLOTS)
    assert beyond  # neighbours without a slot


@pytest.mark.gpu
@pytest.mark.parametrize("form", [lbx.MP_STORED, lbx.MP_RECOMPUTED])
@pytest.mark.parametrize("name", CASES)
def test_layouts_match_restatement(name, form, monkeypatch):
    dims, nat, _ = CASES[name]
    print("mp layout", name, form, flush=True)
    sys.stdout.flush()
    init = lbx.Lattice.__init__

    def with_form(self, *a, **k):
        init(self, *a, **k)
        self.set_mp_coefficients(form)

    monkeypatch.setattr(lbx.Lattice, "__init__", with_form)
    rho, j, _, fields = run_single(dims, nat, lbx.PREC_FP64, None, FEXT, KA, KD, 9)
    nt = lbref.tracer_population(dims, nat, rho, j, FEXT)
    for t in range(3):
        mp = lbref.MP(dims, nat, lbref.interfacial(*dims, nat), nt, rho, 0.01, KA[t], KD[t])
        assert mp.run(9)[0] == 0
        assert np.array_equal(fields[t][0], mp.P)
        if mp.ads:
            assert np.array_equal(fields[t][1], mp.Pa)


@pytest.mark.gpu
@pytest.mark.parametrize("prec", [lbx.PREC_FP32_SHIFT, lbx.PREC_FP32_STORE])
@pytest.mark.parametrize("form", [lbx.MP_STORED, lbx.MP_RECOMPUTED])
@pytest.mark.parametrize("name", CASES)
def test_fp32_tracers_match_restatement(name, form, prec):
    dims, nat, _ = CASES[name]
    print("mp layout fp32", name, form, prec, flush=True)
    with lbx.Lattice(dims, nat, 0.9, precision=prec) as L:
        L.set_mp_coefficients(form)
        L.init_rest(1.0)
        L.equilibrate(FEXT, 0.0, max_steps=12)
        _, rho, j = L.get_state(populations=False)
        v0 = L.mp_init_batch(FEXT, 0.01, KA, KD)
        v = L.mp_run(9)["vacf"].reshape(9, 3, 3)
        fields = [L.mp_get(t) for t in range(3)]
        for t in range(3):
            st, _, P, Pa = lbref.mp_shift(dims, nat, lbref.interfacial(*dims, nat), rho, j, FEXT, 0.01, KA[t], KD[t], 9)
            assert st == 0
            w0 = L.mp_init(FEXT, 0.01, KA[t], KD[t])
            w = L.mp_run(9)["vacf"]
            assert np.array_equal(v0[t], w0) and np.array_equal(v[:, t], w)
            for a, b, ref in zip(fields[t], L.mp_get(), (P, Pa)):
                assert np.array_equal(a, b) and np.array_equal(a, ref)


@pytest.mark.gpu
@pytest.mark.parametrize("mode", [lbx.LAUNCH_GRAPH, lbx.LAUNCH_PERSISTENT])
@pytest.mark.parametrize("prec", [lbx.PREC_FP64, lbx.PREC_FP32_SHIFT, lbx.PREC_FP32_STORE])
def test_batch_of_layouts_equals_single(prec, mode):
    """All kinds in one batch, and those without the general step: VACF and
    D_eff of each are the single lattice's bits."""
    print("mp layout batch", prec, mode, flush=True)
    steps = 11
    for names in (list(CASES), [n for n in CASES if CASES[n][2] != "general"]):
        sizes = [CASES[n][1] for n in names]
        cap = sum(-(-int((s == 0).sum()) // 256) * 256 for s in sizes)
        with lbx.Batch(cap, sum(s.size for s in sizes), len(names), precision=prec) as B:
            B.set_launch_mode(mode)
            ids = [B.add(CASES[n][0], CASES[n][1], 0.9, 1.0, FEXT, 0.0, 0.01, 0.02, 0.01, steps, max_lb_steps=12)
                   for n in names]
            assert None not in ids
            while B.round(8, 8):
                pass
            got = [B.result(i, vacf_rows=steps + 1) for i in ids]
        for n, g in zip(names, got):
            with lbx.Lattice(*CASES[n][:2], 0.9, precision=prec) as L:
                L.init_rest(1.0)
                L.equilibrate(FEXT, 0.0, max_steps=12)
                v0 = L.mp_init(FEXT, 0.01, 0.02, 0.01)
                m = L.mp_run(steps)
                assert np.array_equal(g["vacf"], np.vstack([v0, m["vacf"]])), n
                assert np.array_equal(g["deff"], L.mp_deff()), n


@pytest.mark.gpu
@pytest.mark.parametrize("prec", [lbx.PREC_FP64, lbx.PREC_FP32_SHIFT])
def test_general_instance_does_not_slow_its_batch(prec):
    """The MP time of two open boxes alone and beside a small lattice that needs
    the general step (1.9 times as long when that took every instance to it)."""
    print("mp layout batch time", prec, flush=True)
    dims, steps = (128, 128, 96), 512
    ms = []
    for beside in (0, 1):
        cases = [box(*dims)] * 2 + [CASES["corner_lines"][:2]] * beside
        cap = sum(-(-int((n == 0).sum()) // 256) * 256 for _, n in cases)
        with lbx.Batch(cap, sum(n.size for _, n in cases), len(cases), precision=prec) as B:
            for d, n in cases:
                assert B.add(d, n, 0.9, 1.0, FEXT, 0.0, 0.01, 0.02, 0.01, steps, max_lb_steps=4) is not None
            while B.round(4, 128):
                pass
            ms.append(B.stats()["mp_ms"])
    print("alone / beside a general one, us per step", *[m / steps * 1e3 for m in ms], flush=True)
    assert ms[1] < 1.25 * ms[0]
