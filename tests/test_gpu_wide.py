"""The wide kernel-table classes (N = 2^(IR - s) cells, grids.f:888-951) on the
GPU against the FP64 oracle, class by class: one species at a time on a nest of
patches down to level 7, so a level-l patch holds only the class N = 2^(l - s).
Few particles take the direct walk, many the histogram form in each of its
layouts (masses, kernel columns, kernel planes: N = 2..4, 8 and 16..32 on a
16 x 8 x 8 tile) and the direct walk again beyond them (N >= 64)."""
import numpy as np
import pytest

from asohf_amd import synth
from asohf_amd.geometry import Geometry, background, f32
from oracle import oracle as O

pytestmark = pytest.mark.gpu

BOX, NX, NL = 8.0, 16, 7


def nest():
    """One patch per level, odd sides, each inside the last."""
    rote, rete = background(0.7, 0.3)
    none = [np.zeros(0)] * 6
    b = Geometry(NX, NX, NX, f32(BOX), rote, rete, np.zeros(1, np.int32), *none)
    n, r = [], []
    for l in range(1, NL + 1):
        d = f32(b.dx / f32(2.0) ** (l - 1))
        n.append((18 + l, 21 - l, 17))
        r.append([b.radx[5]] * 3 if l == 1 else [f32(v + (f32(3.0) - f32(1.5)) * d) for v in r[-1]])
    cols = [np.array([v[a] for v in n], np.int32) for a in range(3)]
    rcols = [np.array([v[a] for v in r], np.float32) for a in range(3)]
    return Geometry(NX, NX, NX, f32(BOX), rote, rete, np.array([0] + [1] * NL, np.int32), *cols, *rcols, fdm=f32(0.845))


def snapshot(g, n, species):
    rng = np.random.default_rng(n + species)
    p = []
    for q in range(g.npatch_total):          # around every patch, out to a base cell
        c0 = np.array([g.prx[q], g.pry[q], g.prz[q]], float)
        side = np.array([g.pnx[q], g.pny[q], g.pnz[q]]) * float(g.dx) / 2.0 ** (q + 1)
        p.append(c0 + rng.uniform(-0.3, 1.3, (n // NL, 3)) * side + rng.uniform(-1, 1, (n // NL, 3)) * float(g.dx))
    h = BOX / 2
    p = ((np.concatenate(p) + h) % BOX - h).astype(np.float32)
    p[p >= f32(h)] = -f32(h)
    m = rng.choice(np.array([1.0, 0.5, 2.5], np.float32), len(p))
    esp = np.zeros(9, np.int32)
    esp[species] = len(p)
    return synth.Snapshot(p[:, 0].copy(), p[:, 1].copy(), p[:, 2].copy(), m, esp, g)


@pytest.mark.parametrize("reduction", ["deterministic", "atomic"])
@pytest.mark.parametrize("n", [70, 35000])
@pytest.mark.parametrize("species", [0, 1, 5])
def test_wide_classes_vs_oracle(n, species, reduction):
    import torch

    from asohf_amd.density import DensityBuilder
    g = nest()
    snap = snapshot(g, n, species)
    d1, d11, _ = O.density64(snap, "A")
    off, lev = g.patch_offsets(), g.level_of_patch()
    t = [torch.from_numpy(a).to("cuda:0") for a in (snap.x, snap.y, snap.z, snap.m)]
    b = DensityBuilder(0)
    try:
        for tile in ((8, 8, 8), (16, 8, 8), (16, 16, 8), (16, 16, 16)):
            b.set_tune(tile=tile)
            r = b.density(g, *t, snap.npart_esp, mode="table", reduction=reduction)
            got = r.u11.cpu().numpy()
            for q in range(g.npatch_total):
                ref = d11[off[q]:off[q + 1]]
                # per cell: the FP32 roundings of the kernel values, products and
                # divisions relative to the cell (atomic mode adds n terms in
                # FP32), and half a unit of 2^-29 max(m) for every member's term
                unit = 2.0 ** -29 * float(snap.m.max()) / float(g.denbas(int(lev[q]))) / float(g.fdm)
                rtol = 12 * 2.0 ** -24 + (2.0 ** -24 * n if reduction == "atomic" else 0.0)
                err = np.abs(got[off[q]:off[q + 1]] - ref)
                assert np.all(err <= 0.5 * unit * snap.n + rtol * np.abs(ref)), (tile, q, err.max(), ref.max())
            if reduction == "deterministic":
                again = b.density(g, *t, snap.npart_esp, mode="table")
                assert torch.equal(r.u11, again.u11) and torch.equal(r.grid_mass, again.grid_mass)
    finally:
        b.close()
