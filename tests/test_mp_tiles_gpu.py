"""The tiles of moment propagation (lbx_mp.h) where their layout changes: full
and merged bricks, tiles taken apart because their halo outgrows a brick's, and
lattices that need the general step (neighbours without an LDS slot, or
densities outside the range of the fast quotient).  P, Pa bit for bit and VACF
within 1e-12 of |VACF(0)| (another summation order) against the restatement,
alone and as batch instances, whose VACF equals the single lattice's bits.

layout() restates the grouping, so that each case is known to be the kind it
is meant to be."""
import sys

import numpy as np
import pytest

import lbref
from laboetie_amd import lbx

C = np.array([(1, 0, 0), (-1, 0, 0), (0, 1, 0), (0, -1, 0), (0, 0, 1), (0, 0, -1), (1, 1, 0), (-1, 1, 0), (1, -1, 0),
              (-1, -1, 0), (1, 0, 1), (-1, 0, 1), (1, 0, -1), (-1, 0, -1), (0, 1, 1), (0, -1, 1), (0, 1, -1),
              (0, -1, -1)])


def layout(dims, nat, brick=(8, 8, 4)):
    """(kind, largest halo of the merged tiles) of a lattice cut into `brick`s."""
    lx, ly, lz = dims
    fluid = nat.reshape(lz, ly, lx) == 0
    nb = [-(-n // b) for n, b in zip(dims, brick)]
    cx, cy = min(8, nb[0]), min(8, nb[1])
    walk = [(x0 + x, y0 + y, z) for y0 in range(0, nb[1], cy) for x0 in range(0, nb[0], cx) for z in range(nb[2])
            for y in range(cy) for x in range(cx)]
    nodes = [np.argwhere(fluid[z * brick[2]:(z + 1) * brick[2], y * brick[1]:(y + 1) * brick[1],
                               x * brick[0]:(x + 1) * brick[0]]) + (z * brick[2], y * brick[1], x * brick[0])
             for x, y, z in walk]
    bound = 2 * -(-int(fluid.sum()) // 256)

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

    tiles = group(128)
    if len(tiles) > bound:
        tiles = group(len(walk))
    assert len(tiles) <= bound
    halo = []
    for t in tiles:
        own = {tuple(v) for n in t for v in n}
        out = {((z + c[2]) % lz, (y + c[1]) % ly, (x + c[0]) % lx) for z, y, x in own for c in C} - own
        halo.append(sum(bool(fluid[v]) for v in out))
    apart = sum(len(t) if h > 344 else 1 for t, h in zip(tiles, halo))
    kind = "brick" if max(halo) <= 344 else "apart" if apart <= bound else "general"
    return kind, max(halo)


def pockets(dims, at):
    """Solid but for the nodes `at` (x, y, z arrays)."""
    nat = np.ones(dims[::-1], np.int8)
    nat[at[2], at[1], at[0]] = 0
    return nat.reshape(-1)


def corner_pockets():
    """2x2x2 pockets around every corner of the bricks."""
    dims = (64, 64, 16)
    x, y, z = np.meshgrid(*[np.concatenate([np.arange(0, n, b), np.arange(b - 1, n, b)])
                            for n, b in zip(dims, (8, 8, 4))], indexing="ij")
    return dims, pockets(dims, (x.ravel(), y.ravel(), z.ravel()))


def facing_crosses():
    """Single nodes on the faces of one plane of bricks, each facing a cross of
    five nodes in the next plane."""
    dims = (64, 64, 8)
    x, y = (v.ravel() for v in np.meshgrid(np.arange(1, 62, 3), np.arange(1, 62, 3), indexing="ij"))
    at = [(x, y, np.full_like(x, z)) for z in (0, 3)]
    at += [(x + dx, y + dy, np.full_like(x, z)) for z in (4, 7)
           for dx, dy in ((0, 0), (1, 0), (-1, 0), (0, 1), (0, -1))]
    return dims, pockets(dims, [np.concatenate(v) for v in zip(*at)])


def noise(dims, solid, seed):
    rng = np.random.default_rng(seed)
    nat = (rng.random(int(np.prod(dims))) < solid).astype(np.int8)
    nat[0] = 0
    return dims, nat


def foam():
    """Noise beside an open half."""
    dims = (40, 40, 24)
    rng = np.random.default_rng(3)
    p = np.where(np.arange(24)[:, None, None] < 6, 0.55, 0.0) * np.ones(dims[::-1])
    return dims, (rng.random(dims[::-1]) < p).astype(np.int8).reshape(-1)


CASES = {
    "full_bricks": ((24, 16, 12), np.zeros(24 * 16 * 12, np.int8), "brick"),
    "ragged_merged": (*noise((37, 21, 11), 0.3, 1), "apart"),
    "half_foam": (*foam(), None),
    "corner_pockets": (*corner_pockets(), None),
    "facing_crosses": (*facing_crosses(), "general"),
}


def test_layouts_cover_the_kinds():
    """Every way a lattice can be laid out is among the cases; the general one
    with neighbours beyond the 766 slots as well."""
    kinds = {}
    for name, (dims, nat, want) in CASES.items():
        kind, halo = layout(dims, nat)
        print(name, kind, halo)
        assert want in (None, kind), (name, kind, halo)
        kinds.setdefault(kind, []).append(halo)
    assert set(kinds) == {"brick", "apart", "general"}
    assert max(kinds["general"]) > 766


def run_single(dims, nat, prec, flow, fext, ka, kd, steps):
    with lbx.Lattice(dims, nat, 0.9, precision=prec) as L:
        if flow is None:
            L.init_rest(1.0)
            L.equilibrate(fext, 0.0, max_steps=12)
            v0 = L.mp_init_batch(fext, 0.01, ka, kd)
            _, rho, j = L.get_state(populations=False)
        else:
            rho, j = flow
            v0 = L.mp_init(fext, 0.01, ka[0], kd[0], flow=flow)[None]
        m = L.mp_run(steps)
        v = m["vacf"].reshape(steps, len(ka), 3)
        return rho, j, np.concatenate([v0[None], v]), [L.mp_get(t) for t in range(len(ka))]


def check(dims, nat, rho, j, fext, ka, kd, vacf, fields):
    itf = lbref.interfacial(*dims, nat)
    nt = lbref.tracer_population(dims, nat, rho, j, fext)
    for t in range(len(ka)):
        mp = lbref.MP(dims, nat, itf, nt, rho, 0.01, ka[t], kd[t])
        st, ref = mp.run(len(vacf) - 1)
        assert st == 0
        assert np.abs(vacf[:, t] - ref).max() <= 1e-12 * np.abs(ref[0]).max()
        assert np.array_equal(fields[t][0], mp.P)
        if mp.ads:
            assert np.array_equal(fields[t][1], mp.Pa)


@pytest.mark.gpu
@pytest.mark.parametrize("form", [lbx.MP_STORED, lbx.MP_RECOMPUTED])
@pytest.mark.parametrize("name", CASES)
def test_tiles_match_restatement(name, form, monkeypatch):
    dims, nat, _ = CASES[name]
    print("mp tiles", name, form, flush=True)
    sys.stdout.flush()
    init = lbx.Lattice.__init__

    def with_form(self, *a, **k):
        init(self, *a, **k)
        self.set_mp_coefficients(form)

    monkeypatch.setattr(lbx.Lattice, "__init__", with_form)
    fext, ka, kd = [2e-5, -1e-5, 3e-5], [0.02, 0.0, 0.05], [0.01, 0.0, 0.01]
    rho, j, v, fields = run_single(dims, nat, lbx.PREC_FP64, None, fext, ka, kd, 9)
    check(dims, nat, rho, j, fext, ka, kd, v, fields)


@pytest.mark.gpu
@pytest.mark.parametrize("prec", [lbx.PREC_FP64, lbx.PREC_FP32_SHIFT, lbx.PREC_FP32_STORE])
def test_batch_of_all_layouts_equals_single(prec):
    """All kinds in one batch (so that the general kernel steps every
    instance), then the brick tiles alone: VACF and D_eff of each are the
    single lattice's bits."""
    print("mp tiles batch", prec, flush=True)
    fext, steps = [2e-5, -1e-5, 3e-5], 11
    for names in (list(CASES), ["full_bricks", "ragged_merged", "half_foam"]):
        sizes = [CASES[n][1] for n in names]
        cap = sum(-(-int((s == 0).sum()) // 256) * 256 for s in sizes)
        with lbx.Batch(cap, sum(s.size for s in sizes), len(names), precision=prec) as B:
            ids = [B.add(CASES[n][0], CASES[n][1], 0.9, 1.0, fext, 0.0, 0.01, 0.02, 0.01, steps, max_lb_steps=12)
                   for n in names]
            assert None not in ids
            while B.round(8, 8):
                pass
            got = [B.result(i, vacf_rows=steps + 1) for i in ids]
        for n, g in zip(names, got):
            dims, nat, _ = CASES[n]
            with lbx.Lattice(dims, nat, 0.9, precision=prec) as L:
                L.init_rest(1.0)
                L.equilibrate(fext, 0.0, max_steps=12)
                v0 = L.mp_init(fext, 0.01, 0.02, 0.01)
                m = L.mp_run(steps)
                assert np.array_equal(g["vacf"], np.vstack([v0, m["vacf"]])), n
                assert np.array_equal(g["deff"], L.mp_deff()), n


@pytest.mark.gpu
@pytest.mark.parametrize("scale", [1.0, 2.0 ** 399, 2.0 ** 401, 2.0 ** -401])
def test_densities_outside_the_fast_quotient(scale):
    """Flows with densities at and beyond the range in which the step divides
    by a shared reciprocal (P depends on the ratio of flow to density only)."""
    dims, nat = noise((19, 11, 9), 0.25, 7)
    print("mp tiles density", scale, flush=True)
    rng = np.random.default_rng(5)
    fluid = nat == 0
    rho = np.where(fluid, 1.0 + 0.05 * rng.standard_normal(nat.size), 0.0) * scale
    j = np.where(fluid, 0.01 * rng.standard_normal((3, nat.size)), 0.0) * scale
    fext = [0.0, 0.0, 0.0]
    with lbx.Lattice(dims, nat, 0.9) as L:
        L.set_mp_coefficients(lbx.MP_RECOMPUTED)
        v0 = L.mp_init(fext, 0.01, 0.02, 0.01, flow=(rho, j))
        m = L.mp_run(9)
        fields = [L.mp_get()]
    check(dims, nat, rho, j, fext, [0.02], [0.01], np.concatenate([v0[None, None], m["vacf"][:, None]]), fields)
