"""Projection through its counting and accumulation variants: LDS counters (J <= 8, one or four particles a thread),
global counters (J >= 9), 1024-thread tiles (J <= 6), empty and ragged catalogues.

The sums are integers, so the coefficients do not depend on the order of the particles: bit for bit the same for a
permuted catalogue, whatever bucketing it takes.  Against the oracle: cells, fractions and counts bit for bit, and
coefficients within 1e-12 of the largest plus the resolution of a tile's fixed point: n records of at most
u = max |w| max |phi|^3 each are scaled to fill 2^61, so each of up to n contributions of a cell is rounded to
n u 2^-60 or finer."""

import numpy as np
import pytest

from oracle import projection as oproj

pytestmark = pytest.mark.gpu

BOX = 700.0


@pytest.mark.parametrize("J,n", [(3, 1), (4, 255), (5, 257), (6, 1023), (6, 300_001), (7, 5_000), (8, 262_145),
                                 (8, 999), (9, 3_001)])
@pytest.mark.parametrize("clustered", [False, True])
def test_projection_variants(phi, J, n, clustered):
    import torch
    from pyhermes_amd import kernels
    rng = np.random.default_rng(100 * J + n % 97)
    pos = rng.uniform(0, BOX, size=(n, 3))
    if clustered:  # all in a few tiles, some on cell and box edges
        pos = np.mod(pos * 0.03 + BOX - 0.01 * BOX, BOX)
        pos[::7, 2] = 0.0
    w = rng.normal(size=n)
    print(f"projection J={J} n={n} clustered={clustered}", flush=True)
    out = kernels.project(pos, w, J, BOX, phi, want32=True, want64=True, want_cells=True, want_counts=True)
    mix = rng.permutation(n)
    again = kernels.project(pos[mix], w[mix], J, BOX, phi, want64=True)
    ref, cell, frac = oproj.project_c(pos, w, phi, J, BOX)
    assert torch.equal(out["eps64"], again["eps64"]) and torch.equal(out["eps32"], again["eps32"])
    scale = np.abs(ref).max()
    fixed = n * n * np.abs(w).max() * np.abs(phi).max() ** 3 * 2.0 ** -60
    assert np.abs(out["eps64"].cpu().numpy() - ref).max() <= 1e-12 * scale + fixed
    assert np.abs(out["eps32"].cpu().numpy() - ref).max() <= 2.0 ** -23 * scale + fixed
    assert np.array_equal(out["cell"].cpu().numpy(), cell) and np.array_equal(out["frac"].cpu().numpy(), frac)
    L = 1 << J
    c = np.mod(cell.astype(np.int64), L)
    counts = np.bincount((c[:, 0] * L + c[:, 1]) * L + c[:, 2], minlength=L ** 3).reshape(L, L, L)
    assert np.array_equal(out["counts"].cpu().numpy(), counts)


@pytest.mark.parametrize("J", [5, 9])
def test_empty_and_invalid_catalogues(phi, J):
    import torch
    from pyhermes_amd import kernels
    empty = kernels.project(np.zeros((0, 3)), np.zeros(0), J, BOX, phi, want64=True)
    assert not empty["eps64"].any() and not empty["eps32"].any()
    pos = np.random.default_rng(0).uniform(0, BOX, size=(500, 3))
    good = kernels.project(pos, np.ones(500), J, BOX, phi, want64=True)["eps64"]
    bad = pos.copy()
    bad[499, 1] = np.nan
    with pytest.raises(RuntimeError, match="non-finite"):
        kernels.project(bad, np.ones(500), J, BOX, phi)
    assert torch.equal(kernels.project(pos, np.ones(500), J, BOX, phi, want64=True)["eps64"], good)
