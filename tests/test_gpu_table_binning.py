"""Kernel-table binning through the base grid (each base tile's entries tested
against the patches that can hold a particle of the tile) against the count and
scatter passes over the patch hash: the same entries, so the same fields bit
for bit and the same member and entry counts.  The snapshots put particles of
every species around patches that touch and cross the box's faces, inside the
box, a little outside it and most of a box away (periodic images, which the
binning enumerates one by one), more targets than one LDS batch holds, and a
second call whose particles overflow the first call's capacities."""
import numpy as np
import pytest

from conftest import FIXTURES, load_fixture

from asohf_amd import synth
from asohf_amd.geometry import Geometry, background, f32

pytestmark = pytest.mark.gpu

BOX, NX = 8.0, 20


def geometry(copies):
    rote, rete = background(0.7, 0.3)
    none = [np.zeros(0)] * 6
    b = Geometry(NX, NX, NX, f32(BOX), rote, rete, np.zeros(1, np.int32), *none)
    lvl1 = [((8, 12, 9), (1, 1, 1)), ((16, 7, 20), (NX - 7, 3, 9)), ((2, 33, 5), (9, 2, NX - 2))] * copies
    n = [list(v[0]) for v in lvl1]
    r = [[b.radx[i] for i in v[1]] for v in lvl1]
    for q in range(3):                       # one level-2 patch inside each of the first three
        n.append([5, 6, 3])
        r.append([f32(v + f32(0.5) * f32(b.dx / f32(2.0))) for v in r[q]])
    cols = [np.array([v[a] for v in n], np.int32) for a in range(3)]
    rcols = [np.array([v[a] for v in r], np.float32) for a in range(3)]
    return Geometry(NX, NX, NX, f32(BOX), rote, rete, np.array([0, len(lvl1), 3], np.int32), *cols, *rcols)


def particles(n, seed, outside):
    rng = np.random.default_rng(seed)
    h = BOX / 2
    p = rng.uniform(-h, h, (n, 3))
    p[: n // 3] = rng.choice([-h, h - 1e-6, 0.0], (n // 3, 3)) + rng.uniform(-0.6, 0.6, (n // 3, 3))
    if outside:
        p[: n // 20] += rng.choice([-1.0, 0.0, 1.0], (n // 20, 3)) * 0.9 * BOX
        p = np.clip(p, -1.4 * BOX, 1.4 * BOX)
    else:
        p = np.clip(p, -h, h - 1e-5)
    p = p.astype(np.float32)
    m = rng.choice(np.array([1.0, 0.5], np.float32), n)
    cut = np.sort(rng.integers(0, n, 8))
    esp = np.diff(np.concatenate([[0], cut, [n]])).astype(np.int32)
    return p[:, 0].copy(), p[:, 1].copy(), p[:, 2].copy(), m, esp


def snapshots():
    for name in FIXTURES:
        s = load_fixture(name)[0]
        yield name, s.geom, [(s.x, s.y, s.z, s.m, s.npart_esp)]
    for copies in (1, 30):
        g = geometry(copies)
        for outside in (False, True):
            yield (f"faces x{copies} outside {outside}", g,
                   [particles(9000, 1, outside), particles(9000, 2, outside), particles(401, 3, outside)])


@pytest.mark.parametrize("reduction", ["deterministic", "atomic"])
def test_base_grid_binning_equals_hash_binning(monkeypatch, reduction):
    import torch

    from asohf_amd.density import DensityBuilder
    monkeypatch.setenv("ASOHF_TSC_BINNING", "hash")
    hashed = DensityBuilder(0)
    monkeypatch.delenv("ASOHF_TSC_BINNING")
    based = DensityBuilder(0)
    try:
        for name, g, sets in snapshots():
            for k, (x, y, z, m, esp) in enumerate(sets):
                for chunk in (64, 4096):
                    print(f"case table binning: {name} set {k} chunk {chunk} {reduction}", flush=True)
                    t = [torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0") for a in (x, y, z, m)]
                    got = []
                    for b in (based, hashed):
                        b.set_tune(chunk=chunk)
                        r = b.density(g, *t, esp, mode="table", reduction=reduction)
                        st = b.stats()
                        got.append((r.u1, r.u11[:int(g.patch_cells().sum())], r.grid_mass, st["n_pairs"], st["n_entries"]))
                    assert got[0][3:] == got[1][3:], (name, k)
                    for u, v in zip(got[0][:3], got[1][:3]):
                        if reduction == "deterministic":
                            assert torch.equal(u, v), (name, k)
                        else:
                            # FP32 sums in another order: n roundings of 2^-24
                            assert torch.allclose(u, v, rtol=len(m) * 2.0 ** -24, atol=0.0), (name, k)
    finally:
        hashed.close()
        based.close()


def test_positions_the_wrap_rejects_stay_rejected():
    import torch

    from asohf_amd import _lib
    from asohf_amd.density import DensityBuilder
    g = geometry(1)
    x, y, z, m, esp = particles(500, 4, False)
    b = DensityBuilder(0)
    try:
        for bad in (np.float32(2.1 * BOX), np.float32(np.nan), np.float32(-1e30)):
            xb = x.copy()
            xb[77] = bad
            t = [torch.from_numpy(a).to("cuda:0") for a in (x, y, z, m)]
            b.density(g, *t, esp, mode="table")
            t[0] = torch.from_numpy(xb).to("cuda:0")
            with pytest.raises(_lib.AsohfError):
                b.density(g, *t, esp, mode="table")
    finally:
        b.close()
