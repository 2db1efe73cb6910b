"""The exchange between deposit tiles, on the GPU, against the FP64 oracle.

An entry is deposited by the one tile that holds its centre cell; what its
stencil spills over the tile's border reaches the neighbouring tiles through
their halo cells.  The cases put particles on both sides of every tile border
and of the periodic wrap, on base grids of one and several tiles per axis with
full, partial and one-cell last tiles, and on patches whose sides leave the
same remainders, with particles up to a cell outside the patch."""
import numpy as np
import pytest

from asohf_amd import synth
from asohf_amd.geometry import Geometry, background, f32
from oracle import oracle as O

pytestmark = pytest.mark.gpu

BOX = 10.0
TILES = ((8, 8, 8), (16, 8, 8), (16, 16, 8), (16, 16, 16))


def snapshot(nx, sides):
    """nx^3 base grid and, where they fit, one level-1 patch of each side; the
    particles lie around every cell centre's faces near tile borders."""
    rote, rete = background(0.7, 0.3)
    none = [np.zeros(0)] * 6
    base = Geometry(nx, nx, nx, f32(BOX), rote, rete, np.zeros(1, np.int32), *none)
    n = [tuple(s) for s in sides]
    pr = [[base.radx[2 + 3 * k % max(nx - 2, 1)] for _ in range(3)] for k in range(len(n))]
    cols = [np.array([v[a] for v in n], np.int32) for a in range(3)]
    rcols = [np.array([v[a] for v in pr], np.float32) for a in range(3)]
    g = base if not n else Geometry(nx, nx, nx, f32(BOX), rote, rete, np.array([0, len(n)], np.int32), *cols, *rcols,
                                    fdm=f32(0.845))
    rng = np.random.default_rng(nx)
    h = BOX / 2
    pos = [rng.uniform(-h, h, (3000, 3))]
    edge = np.array([0.0, 1e-6, BOX / nx, 8 * BOX / nx, 16 * BOX / nx, BOX - 1e-6]) - h
    edge = edge[edge < h]
    pos.append(rng.choice(edge, (1500, 3)) + rng.uniform(-1, 1, (1500, 3)) * 1.2 * BOX / nx)
    p = np.concatenate(pos)
    p = ((p + h) % BOX - h).astype(np.float32)
    p[p >= f32(h)] = -f32(h)
    m = rng.choice(np.array([1.0, 0.25, 3.0], np.float32), len(p))
    esp = np.zeros(9, np.int32)
    esp[0], esp[1] = len(p) // 2, len(p) - len(p) // 2
    return synth.Snapshot(p[:, 0].copy(), p[:, 1].copy(), p[:, 2].copy(), m, esp, g)


CASES = [(3, ()), (5, ()), (8, ((1, 2, 3),)), (9, ((8, 9, 7),)), (16, ((16, 17, 15), (2, 8, 1))),
         (17, ((18, 16, 8), (7, 1, 33))), (33, ((32, 9, 25), (1, 1, 1), (17, 24, 16)))]


@pytest.mark.parametrize("mode", ["tsc", "table"])
@pytest.mark.parametrize("nx,sides", CASES)
def test_spilled_stencils_reach_their_cells(nx, sides, mode):
    import torch

    from asohf_amd.density import DensityBuilder
    snap = snapshot(nx, sides)
    g = snap.geom
    d = O.density64(snap, "A" if mode == "table" else "B")
    # FP32 weights, products and divisions: 9 roundings of 2^-24; every term
    # and every particle's remainder within one and 13 units of 2^-29 max(m)
    unit = 2.0 ** -29 * float(snap.m.max()) / float(g.denbas(g.nl)) / float(g.fdm)
    atol, rtol = 14 * unit * snap.n, 9 * 2.0 ** -24
    t = [torch.from_numpy(a).to("cuda:0") for a in (snap.x, snap.y, snap.z, snap.m)]
    b = DensityBuilder(0)
    first = None
    try:
        for tile in TILES:
            for chunk in (64, 4096):
                b.set_tune(tile=tile, chunk=chunk)
                r = b.density(g, *t, snap.npart_esp, mode=mode)
                got = [v.cpu().numpy() for v in (r.u1, r.u11[:int(g.patch_cells().sum())], r.grid_mass)]
                for u, ref in zip(got[:1 + (g.npatch_total > 0)], d):
                    assert np.all(np.abs(u.ravel() - ref.ravel()) <= atol + rtol * np.abs(ref.ravel())), (tile, chunk)
                # every particle deposits exactly its mass (a multiple of the unit) on the base grid
                assert got[2][0] == snap.m.astype(np.float64).sum(), (tile, chunk)
                first = first or got
                assert np.array_equal(got[0], first[0]), (tile, chunk)
                if mode == "tsc":
                    assert all(np.array_equal(u, v) for u, v in zip(got, first)), (tile, chunk)
    finally:
        b.close()


@pytest.mark.parametrize("mode", ["tsc", "table"])
@pytest.mark.parametrize("nx,sides", CASES)
def test_atomic_sums_reach_the_same_cells(nx, sides, mode):
    """Atomic mode sums FP32 terms: table mode then keeps an entry in every tile
    a stencil touches (two images of one tile where the last tile of a
    two-tile axis is one cell wide)."""
    import torch

    from asohf_amd.density import DensityBuilder
    snap = snapshot(nx, sides)
    d = O.density64(snap, "A" if mode == "table" else "B")
    rtol = (9 + snap.n) * 2.0 ** -24   # n FP32 sums
    t = [torch.from_numpy(a).to("cuda:0") for a in (snap.x, snap.y, snap.z, snap.m)]
    b = DensityBuilder(0)
    try:
        for tile in TILES:
            b.set_tune(tile=tile)
            r = b.density(snap.geom, *t, snap.npart_esp, mode=mode, reduction="atomic")
            got = [r.u1.cpu().numpy(), r.u11[:int(snap.geom.patch_cells().sum())].cpu().numpy()]
            for u, ref in [(u, ref) for u, ref in zip(got, d) if ref.size and u.size]:
                # atol: the FP32 weights of a far corner cell keep few digits (1.5 - b cancels)
                assert np.all(np.abs(u.ravel() - ref.ravel()) <= 2.0 ** -20 * ref.max() + rtol * ref.ravel()), tile
    finally:
        b.close()


@pytest.mark.parametrize("masses", [(1.0,), (1.0, 0.25), (3e-7, 1.0, 0.1, 0.7)])
def test_counted_masses_equal_single_deposits(masses):
    """Table mode counts the entries of an item's first mass per cell and
    deposits the others one by one: the same integers whichever mass comes
    first, so the fields do not depend on the particle order or the item size,
    and the base grid keeps the quantised mass exactly."""
    import torch

    from asohf_amd.density import DensityBuilder
    snap = snapshot(17, ((18, 16, 8), (7, 1, 33)))
    rng = np.random.default_rng(len(masses))
    m = rng.choice(np.array(masses, np.float32), snap.n)
    half = int(snap.npart_esp[0])
    q = np.rint(m.astype(np.float64) * 2.0 ** (30 - int(np.frexp(np.float32(m.max()))[1])))
    b = DensityBuilder(0)
    first = None
    try:
        for k in range(3):
            # another order within each species block
            o = np.concatenate([rng.permutation(half), half + rng.permutation(snap.n - half)]) if k else np.arange(snap.n)
            t = [torch.from_numpy(a[o]).to("cuda:0") for a in (snap.x, snap.y, snap.z, m)]
            for chunk in (64, 4096):
                b.set_tune(chunk=chunk)
                r = b.density(snap.geom, *t, snap.npart_esp, mode="table")
                got = [v.cpu().numpy() for v in (r.u1, r.u11, r.grid_mass)]
                assert got[2][0] == q.sum() / 2.0 ** (30 - int(np.frexp(np.float32(m.max()))[1]))
                first = first or got
                assert np.array_equal(got[0], first[0]) and np.array_equal(got[1], first[1])
    finally:
        b.close()
