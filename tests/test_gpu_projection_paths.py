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


def test_catalogue_too_large_to_keep_slots(phi):
    """2^24 + 77 particles (more than 2 GiB of records at worst): slots are not kept, the fill counts again and the
    records are sized after the count.  Counts bit for bit, the same coefficients for a permuted catalogue, and within
    the fixed-point resolution of the contributions a cell can get (those of the particles of 27 cells)."""
    import torch
    from pyhermes_amd import kernels
    J, n = 5, (1 << 24) + 77
    L = 1 << J
    gen = torch.Generator(device="cuda").manual_seed(5)
    pos = torch.rand((n, 3), generator=gen, device="cuda", dtype=torch.float64) * BOX
    w = torch.rand(n, generator=gen, device="cuda", dtype=torch.float64) + 0.5
    kernels.release_workspaces()
    print(f"projection J={J} n={n} without slots", flush=True)
    out = kernels.project(pos, w, J, BOX, phi, want64=True, want_counts=True)
    mix = torch.randperm(n, generator=gen, device="cuda")
    again = kernels.project(pos[mix], w[mix], J, BOX, phi, want64=True)
    assert torch.equal(out["eps64"], again["eps64"]) and torch.equal(out["eps32"], again["eps32"])
    s = pos * (L / BOX)
    c = torch.floor(s)
    f = torch.clamp(((s - c) * 1024).long(), max=1023)
    c = c.long()
    index = lambda a, b, e: (((c[:, 0] - a) % L) * L + (c[:, 1] - b) % L) * L + (c[:, 2] - e) % L
    counts = torch.bincount(index(0, 0, 0), minlength=L ** 3).view(L, L, L)
    assert torch.equal(out["counts"].long(), counts)
    ph = kernels.as_device(phi, torch.float64)
    ref = torch.zeros(L ** 3, dtype=torch.float64, device="cuda")
    for a in range(3):
        for b in range(3):
            for e in range(3):
                ref.index_add_(0, index(a, b, e), w * ph[f[:, 0] + 1024 * a] * ph[f[:, 1] + 1024 * b] * ph[f[:, 2] + 1024 * e])
    near = 27.0 * float(counts.max())
    fixed = near * n * float(w.max()) * np.abs(phi).max() ** 3 * 2.0 ** -60
    # index_add sums in an order of its own: near terms of at most max |ref| size, each rounded
    assert float((out["eps64"].view(-1) - ref).abs().max()) <= (1e-12 + near * 2.0 ** -53) * float(ref.abs().max()) + fixed


@pytest.mark.parametrize("J,n", [(5, 30_001), (8, 262_145), (9, 30_001)])
def test_capture_without_room_for_slots(phi, J, n):
    """A capture that finds the records' room but not the slots' counts again in the fill: bit for bit the eager result
    (LDS counters and slots), on every replay."""
    import torch
    from pyhermes_amd import _lib, kernels
    gen = torch.Generator(device="cuda").manual_seed(J)
    L = 1 << J
    big = torch.rand(((1 << 24) + 1, 3), generator=gen, device="cuda", dtype=torch.float64) * BOX
    pos, w = big[:n].contiguous(), torch.randn(n, generator=gen, device="cuda", dtype=torch.float64)
    ph = kernels.as_device(phi, torch.float64)
    eps = torch.empty((L, L, L), dtype=torch.float64, device="cuda")
    print(f"captured projection J={J} n={n} without slots", flush=True)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        kernels.release_workspaces()
        kernels.project(big, torch.ones(big.shape[0], dtype=torch.float64, device="cuda"), 5, BOX, phi)  # records, no slots
        kernels.project(pos[:9].contiguous(), w[:9].contiguous(), J, BOX, phi)  # the level's tiles, nine particles' slots
        kernels.capture_begin()
        try:
            _lib.call("hermes_project", _lib.context(), pos.data_ptr(), w.data_ptr(), n, J, BOX, ph.data_ptr(), ph.numel(),
                      1024, float(np.abs(phi).max()), None, eps.data_ptr(), None, None, None)
        finally:
            graph = kernels.capture_end()
        got = []
        for _ in range(3):
            eps.fill_(np.nan)
            kernels.graph_launch(graph)
            torch.cuda.synchronize()
            assert kernels.read_errors() == 0
            got.append(eps.clone())
        kernels.graph_destroy(graph)
        want = kernels.project(pos, w, J, BOX, phi, want64=True)["eps64"]
    assert all(torch.equal(g, want) for g in got)


def test_refused_workspace_leaves_no_error_behind(phi):
    """A call whose records cannot be had fails with work in flight that meets an invalid position; the next call must
    be refused neither for the allocation's error nor for that position."""
    import torch
    from pyhermes_amd import kernels
    J, n = 5, 1 << 24
    gen = torch.Generator(device="cuda").manual_seed(7)
    pos = torch.rand((n, 3), generator=gen, device="cuda", dtype=torch.float64) * BOX
    pos[n // 2, 1] = float("inf")
    w = torch.ones(n, dtype=torch.float64, device="cuda")
    good, gw = pos[:4096].clone(), w[:4096].clone()
    want = kernels.project(good, gw, J, BOX, phi, want64=True)["eps64"]
    kernels.release_workspaces()
    torch.cuda.empty_cache()
    print("projection with its records refused", flush=True)
    fill, chunk = [torch.empty(int(0.98 * torch.cuda.mem_get_info()[0]), dtype=torch.uint8, device="cuda")], 1 << 28
    with pytest.raises(torch.cuda.OutOfMemoryError):
        while True:
            fill.append(torch.empty(chunk, dtype=torch.uint8, device="cuda"))
    del fill[-5:]  # 1.25 GiB for the slots and the tiles; the records ask for 2.5
    torch.cuda.empty_cache()
    torch.cuda._sleep(30_000_000)
    with pytest.raises(RuntimeError, match="hermes_project failed .*hipMalloc of .* for workspace slot"):
        kernels.project(pos, w, J, BOX, phi)
    got = kernels.project(good, gw, J, BOX, phi, want64=True)["eps64"]
    del fill
    kernels.release_workspaces()
    torch.cuda.empty_cache()
    assert torch.equal(got, want)
