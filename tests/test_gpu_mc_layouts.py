"""The Monte-Carlo kernels on every grid layout they read: plain and 16-byte aligned grids, grids at odd 8-byte
offsets, bricked copies (L >= 128 with enough points), waves that are not full.

Reference: the oracle on the same draws.  Sums agree to the resolution of the fixed-point accumulators (1e-9, as
for the existing sizes) and the triplet means to FP64 rounding (1e-12); counts bit for bit."""

import numpy as np
import pytest

from oracle import mc as omc

pytestmark = pytest.mark.gpu


def _grid(L, seed):
    return np.random.default_rng(seed).lognormal(0.0, 0.5, size=(L, L, L)) - 1.1


def _device(a, offset):
    """The grid on the device, its first element `offset` doubles into an allocation."""
    import torch
    buf = torch.empty(a.size + offset, dtype=torch.float64, device="cuda")
    t = buf[offset:].view(a.shape)
    t.copy_(torch.from_numpy(a))
    assert t.data_ptr() % 16 == 8 * (offset % 2)
    return t


@pytest.mark.parametrize("L,n,offset", [(32, 1001, 0), (32, 1001, 1), (128, 1001, 1), (128, 90_001, 0), (128, 90_001, 1)])
@pytest.mark.parametrize("same", [True, False])
def test_binned_sampler_layouts(phi, L, n, offset, same):
    from pyhermes_amd import kernels
    nbins, r1r, r2r, seed = (3, 4, 5), (1.5, 9.0), (2.0, 0.3 * L), 17
    g = [_grid(L, 1)] * 3 if same else [_grid(L, s) for s in (1, 2, 3)]
    gd = [_device(g[0], offset)] * 3 if same else [_device(a, offset) for a in g]
    print(f"binned layouts L={L} n={n} offset={offset} same={same}", flush=True)
    ref = omc.binned_sampler(*g, phi, nbins, r1r, r2r, n, seed)
    got = kernels.mc_binned(*gd, phi, nbins, r1r, r2r, n, seed)
    assert np.array_equal(got[2], ref[2])
    for a, b in zip(got[:2], ref[:2]):
        np.testing.assert_allclose(a, b, rtol=1e-9, atol=1e-9 * np.abs(b).max())


@pytest.mark.parametrize("L,n,n_rot,offset", [(16, 1, 1, 0), (64, 777, 3, 1), (128, 65, 2, 0), (128, 40_003, 9, 0),
                                             (128, 40_003, 9, 1)])
def test_triplet_layouts(phi, L, n, n_rot, offset):
    import torch
    from pyhermes_amd import kernels
    g2, g3 = _grid(L, 4), _grid(L, 5)
    rng = np.random.default_rng(n)
    spos = rng.uniform(-2.0 * L, 3.0 * L, size=(n, 3))
    n1, abc = rng.normal(size=n), rng.random((n_rot, 3))
    print(f"triplet layouts L={L} n={n} rot={n_rot} offset={offset}", flush=True)
    got = kernels.mc_triplet_box(0.2 * L, 0.35 * L, -0.3, kernels.as_device(spos, torch.float64),
                                 kernels.as_device(n1, torch.float64), abc, _device(g2, offset), _device(g3, offset), phi)
    ref, mag = 0.0, 0.0
    for a, b, c in abc:
        o = omc.triangle_offsets(0.2 * L, 0.35 * L, -0.3, 2 * np.pi * a, 2 * b - 1, 2 * np.pi * c)
        t = n1 * omc.interpolate(g2, spos, phi, o[:3]) * omc.interpolate(g3, spos, phi, o[3:])
        ref, mag = ref + t.sum(), mag + np.abs(t).sum()
    assert abs(got - ref / (n * n_rot)) <= 1e-12 * mag / (n * n_rot)


def test_bricks_keep_non_finite_cells_apart(phi):
    """A NaN or an infinite cell reaches the triangles whose neighbourhoods hold it and no other."""
    import torch
    from pyhermes_amd import kernels
    L, n = 128, 140_000
    g = _grid(L, 6)
    bad = g.copy()
    bad[5, 6, 7], bad[70, 3, 2] = np.nan, np.inf
    rng = np.random.default_rng(3)
    spos = rng.uniform(0, L, size=(n, 3))
    abc = rng.random((1, 3))
    o = omc.triangle_offsets(9.0, 14.0, 0.2, *(2 * np.pi * abc[0, 0], 2 * abc[0, 1] - 1, 2 * np.pi * abc[0, 2]))
    hit = np.zeros(n, bool)
    for k in (0, 3):
        c = np.floor(spos + o[k:k + 3]).astype(int)
        for cell in ((5, 6, 7), (70, 3, 2)):
            hit |= np.all((c - np.array(cell)) % L <= 2, axis=1)
    assert 0 < hit.sum() < 200
    n1 = np.where(hit, 0.0, 1.0)
    args = (9.0, 14.0, 0.2)
    clean = np.where(hit[:, None], spos[~hit][0], spos)  # the centres that meet a bad cell moved away, weight 0
    dev = lambda a: kernels.as_device(a, torch.float64)
    want = kernels.mc_triplet_box(*args, dev(clean), dev(n1), abc, dev(g), dev(g), phi)
    got = kernels.mc_triplet_box(*args, dev(clean), dev(n1), abc, dev(bad), dev(bad), phi)
    assert np.isfinite(got) and got == want
    assert not np.isfinite(kernels.mc_triplet_box(*args, dev(spos), dev(n1 * 0 + 1), abc, dev(bad), dev(bad), phi))


@pytest.mark.parametrize("level,offset", [(9, 0), (9, 1), (11, 0), (4, 0)])
def test_triplet_with_another_table_resolution(level, offset):
    """2^level samples of the scaling function to a cell instead of 1024, through the C entry: the table is read
    with the caller's resolution (a grid and point count that take the bricks at 1024)."""
    import ctypes
    from oracle.scaling import sample_scaling_function
    from pyhermes_amd import _lib, kernels
    import torch
    L, n, n_rot, res = 128, 40_003, 9, 1 << level
    phi = sample_scaling_function("db2", level)
    assert phi.size == 3 * res
    g2, g3 = _grid(L, 4), _grid(L, 5)
    rng = np.random.default_rng(level)
    spos = rng.uniform(-2.0 * L, 3.0 * L, size=(n, 3))
    n1, abc = rng.normal(size=n), rng.random((n_rot, 3))
    dev = [kernels.as_device(a, torch.float64) for a in (spos, n1, phi)]
    gd = [_device(g2, offset), _device(g3, offset)]
    got = np.zeros(1)
    dp = ctypes.POINTER(ctypes.c_double)
    print(f"triplet with {res} samples to a cell, offset={offset}", flush=True)
    _lib.call("hermes_mc_triplet_box", _lib.context(), 7, 0.2 * L, 0.35 * L, -0.3, dev[0].data_ptr(), dev[1].data_ptr(),
              n, n_rot, abc.ctypes.data_as(dp), gd[0].data_ptr(), gd[1].data_ptr(), dev[2].data_ptr(), res,
              got.ctypes.data_as(dp))
    ref, mag = 0.0, 0.0
    for a, b, c in abc:
        o = omc.triangle_offsets(0.2 * L, 0.35 * L, -0.3, 2 * np.pi * a, 2 * b - 1, 2 * np.pi * c)
        t = n1 * omc.interpolate(g2, spos, phi, o[:3], res) * omc.interpolate(g3, spos, phi, o[3:], res)
        ref, mag = ref + t.sum(), mag + np.abs(t).sum()
    assert abs(got[0] - ref / (n * n_rot)) <= 1e-12 * mag / (n * n_rot)


@pytest.mark.parametrize("n,offset,same", [(200_003, 0, True), (200_003, 1, False), (262_145, 0, True), (400_001, 1, True)])
def test_binned_sampler_rounds(phi, n, offset, same):
    """Sample counts at both sides of the rule for bricks: a round of waves filled by three quarters (bricks), one
    sample more than a round (plain), a round and a half (bricks)."""
    from pyhermes_amd import kernels
    L, nbins, r1r, r2r, seed = 128, (3, 4, 5), (1.5, 9.0), (2.0, 38.0), 23
    g = [_grid(L, 1)] * 3 if same else [_grid(L, s) for s in (1, 2, 3)]
    gd = [_device(g[0], offset)] * 3 if same else [_device(a, offset) for a in g]
    print(f"binned rounds n={n} offset={offset} same={same}", flush=True)
    ref = omc.binned_sampler(*g, phi, nbins, r1r, r2r, n, seed)
    got = kernels.mc_binned(*gd, phi, nbins, r1r, r2r, n, seed)
    assert np.array_equal(got[2], ref[2])
    for a, b in zip(got[:2], ref[:2]):
        np.testing.assert_allclose(a, b, rtol=1e-9, atol=1e-9 * np.abs(b).max())


@pytest.mark.parametrize("n", [300_000, 400_000])
def test_non_finite_cells_stay_apart_at_both_layouts(phi, n):
    """Three quarters of a round of waves (bricks) and one that is just over (plain): a NaN or an infinite cell reaches
    the triangles whose neighbourhoods hold it and no other."""
    from pyhermes_amd import kernels
    import torch
    L = 128
    g = _grid(L, 8)
    bad = g.copy()
    bad[5, 6, 7], bad[70, 3, 2] = np.nan, np.inf
    rng = np.random.default_rng(4)
    spos, abc = rng.uniform(0, L, size=(n, 3)), rng.random((1, 3))
    args = (9.0, 14.0, 0.2)
    o = omc.triangle_offsets(*args, *(2 * np.pi * abc[0, 0], 2 * abc[0, 1] - 1, 2 * np.pi * abc[0, 2]))
    hit = np.zeros(n, bool)
    for k in (0, 3):
        c = np.floor(spos + o[k:k + 3]).astype(int)
        for cell in ((5, 6, 7), (70, 3, 2)):
            hit |= np.all((c - np.array(cell)) % L <= 2, axis=1)
    assert 0 < hit.sum() < 300
    clean = np.where(hit[:, None], spos[~hit][0], spos)
    n1 = np.where(hit, 0.0, 1.0)
    dev = lambda a: kernels.as_device(a, torch.float64)
    print(f"non-finite cells n={n}", flush=True)
    want = kernels.mc_triplet_box(*args, dev(clean), dev(n1), abc, dev(g), dev(g), phi)
    got = kernels.mc_triplet_box(*args, dev(clean), dev(n1), abc, dev(bad), dev(bad), phi)
    assert np.isfinite(got) and got == want
    assert not np.isfinite(kernels.mc_triplet_box(*args, dev(spos), dev(n1 * 0 + 1), abc, dev(bad), dev(bad), phi))


@pytest.mark.parametrize("J", [9, 10])
def test_triplet_on_the_largest_grids(phi, J):
    """1.7e7 triangles on a 512^3 grid (bricks: 1 GiB of copies) and a 1024^3 one (its copy would pass 4 GiB: read as
    it is), against gathers in torch."""
    import torch
    from pyhermes_amd import kernels
    L, n, n_rot = 1 << J, (1 << 18) + 3, 64
    gen = torch.Generator(device="cuda").manual_seed(J)
    g = torch.randn((L, L, L), generator=gen, device="cuda", dtype=torch.float64)
    spos = torch.rand((n, 3), generator=gen, device="cuda", dtype=torch.float64) * L
    n1 = torch.randn(n, generator=gen, device="cuda", dtype=torch.float64)
    abc = np.random.default_rng(J).random((n_rot, 3))
    ph = kernels.as_device(phi, torch.float64)

    def value(s):
        c = torch.floor(s)
        f = torch.clamp(((s - c) * 1024).long(), max=1023)
        c = c.long()
        out = torch.zeros(n, dtype=torch.float64, device="cuda")
        for a in range(3):
            for b in range(3):
                for e in range(3):
                    i = (((c[:, 0] - a) % L) * L + (c[:, 1] - b) % L) * L + (c[:, 2] - e) % L
                    out += g.view(-1)[i] * ph[f[:, 0] + 1024 * a] * ph[f[:, 1] + 1024 * b] * ph[f[:, 2] + 1024 * e]
        return out

    args = (0.02 * L, 0.05 * L, 0.4)
    print(f"triplet J={J}", flush=True)
    got = kernels.mc_triplet_box(*args, spos, n1, abc, g, g, phi)
    ref, mag = 0.0, 0.0
    for a, b, c in abc:
        o = torch.from_numpy(omc.triangle_offsets(*args, 2 * np.pi * a, 2 * b - 1, 2 * np.pi * c)).cuda()
        t = n1 * value(spos + o[:3]) * value(spos + o[3:])
        ref, mag = ref + float(t.sum()), mag + float(t.abs().sum())
    kernels.release_workspaces()
    assert abs(got - ref / (n * n_rot)) <= 1e-12 * mag / (n * n_rot)
