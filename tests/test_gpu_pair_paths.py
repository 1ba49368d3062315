"""The grouped pair-reduction kernels against the general one on the same spectra.

A sphere descriptor added to a list sends the whole list through the general kernel, which evaluates every
window at every alias: the reference here.  Tolerance: |K| <= 1 and the sums are FP64, so both differ from the
exact value by the phase error 2 pi |a| R / L * 2^-53 < 1e-13 (arguments below 1000) and, with rotated phases,
by 2 ulps per radius, each times sum |F1 F2| <= scale; 1e-12 of scale covers them.
"""

import numpy as np
import pytest

from oracle import scaling

pytestmark = pytest.mark.gpu


def _spectra(phi, J, dtype, seed):
    import torch
    from pyhermes_amd import kernels
    L = 1 << J
    gen = torch.Generator(device="cuda").manual_seed(seed)
    f1 = torch.randn((L, L, L), generator=gen, device="cuda", dtype=torch.float64)
    f2 = f1 + 0.5 * torch.randn((L, L, L), generator=gen, device="cuda", dtype=torch.float64)
    P = kernels.as_device(scaling.fourier_power_spectrum(phi, 0, 1, L, 1024), torch.float64)
    scale = float((f1.square().mean() * f2.square().mean()).sqrt()) * L ** 6
    return kernels.rfftn(f1.to(dtype)), kernels.rfftn(f2.to(dtype)), P, scale


def _compare(phi, J, dtype, descs, seed):
    import torch
    from pyhermes_amd import kernels
    F1, F2, P, scale = _spectra(phi, J, dtype, seed)
    got = kernels.pair_reduce(F1, F2, P, descs)
    again = kernels.pair_reduce(F1, F2, P, descs)
    np.testing.assert_array_equal(got, again)
    G1, G2 = F1.to(torch.complex128), F2.to(torch.complex128)
    ref = kernels.pair_reduce(G1, G2, P, descs + [kernels.window_desc("sphere", 2.0)])[:-1]
    assert np.abs(got - ref).max() <= 1e-12 * scale, np.abs(got - ref).max() / scale


RADII = {"linear": lambda L: np.linspace(0.02 * L, 0.3 * L, 7), "uneven": lambda L: np.array([0.0, 0.3, 1.7, 0.31 * L]),
         "one": lambda L: np.array([2.5]), "from_zero": lambda L: np.linspace(0.0, 0.4 * L, 5)}


@pytest.mark.parametrize("J", [1, 2, 3, 5, 7, 8])
@pytest.mark.parametrize("spacing", sorted(RADII))
@pytest.mark.parametrize("ells,dtype", [((0,), "float64"), ((0, 2, 4), "float64"), ((2, 4), "float32"),
                                        ((0, 6, 10), "float32")])
def test_radial_kernel_matches_general(phi, J, spacing, ells, dtype):
    """Shells and multipoles: blocks of 4 (J < 8) and 8, rotated and direct phases, radii down to 0 (series)."""
    import torch
    from pyhermes_amd import kernels
    descs = [kernels.window_desc("shell_multipole", R, l=l) if l else kernels.window_desc("shell", R)
             for l in ells for R in RADII[spacing](1 << J)]
    print(f"radial J={J} {spacing} l={ells} {dtype}", flush=True)
    _compare(phi, J, getattr(torch, dtype), descs, 100 + J)


@pytest.mark.parametrize("J,axis,n_windows,dtype", [(1, 2, 3, "float64"), (3, 0, 16, "float64"), (4, 1, 17, "float32"),
                                                    (5, 2, 70, "float64"), (6, 0, 33, "float32"), (6, 1, 1, "float64"),
                                                    (7, 2, 100, "float64"), (8, 1, 5, "float64")])
def test_axis_line_of_sight_kernel_matches_general(phi, J, axis, n_windows, dtype):
    """Ring / disk / cylshell / cylinder windows along one axis (tiles of 16 windows and 16 positions with
    remainders, several window groups): Bessel arguments from 0 through all three ranges."""
    import torch
    from pyhermes_amd import kernels
    L = 1 << J
    rng = np.random.default_rng(J)
    types = ("ring", "disk", "cylshell", "cylinder")
    descs = [kernels.window_desc(types[i % 4], 0.45 * L * rng.random() if i else 0.0, 0.4 * L * rng.random() if i != 2
                                 else 0.0, axis=axis) for i in range(n_windows)]
    print(f"line of sight J={J} axis={axis} n={n_windows} {dtype}", flush=True)
    _compare(phi, J, getattr(torch, dtype), descs, 200 + J)


def test_mixed_axes_keep_the_general_kernel(phi):
    import torch
    from pyhermes_amd import kernels
    F1, F2, P, scale = _spectra(phi, 5, torch.float64, 9)
    descs = [kernels.window_desc("ring", 3.0, 1.0 + i, axis=i) for i in range(3)]
    got = kernels.pair_reduce(F1, F2, P, descs)
    one = np.array([kernels.pair_reduce(F1, F2, P, [d])[0] for d in descs])
    assert np.abs(got - one).max() <= 1e-12 * scale


@pytest.mark.parametrize("J,n,ells,dtype", [(2, 5, (0,), "float32"), (3, 30, (0, 2), "float64"), (4, 9, (0, 10), "float32"),
                                            (5, 31, (0,), "float64"), (6, 30, (0,), "float32"), (6, 13, (2, 4), "float64")])
def test_radial_kernel_with_split_radii(phi, J, n, ells, dtype):
    """Unevenly spaced radii on small grids, split over workgroups (groups of one and of several steps, a ragged last
    one); the first radius carries one order only, so the groups' channel counts differ."""
    import torch
    from pyhermes_amd import kernels
    R = np.geomspace(0.02, 0.4, n) * (1 << J)
    descs = [kernels.window_desc("shell_multipole", r, l=l) if l else kernels.window_desc("shell", r)
             for l in ells for r in (R[1:] if l == ells[-1] and len(ells) > 1 else R)]
    print(f"radial split J={J} n={n} l={ells} {dtype}", flush=True)
    _compare(phi, J, getattr(torch, dtype), descs, 300 + J)


def test_line_of_sight_tables_beyond_the_default_lds(phi):
    """L = 1024: 70 KB of staged powers, above the dynamic LDS a kernel gets unasked.  Radii and heights keep the
    arguments below 1000."""
    import torch
    from pyhermes_amd import kernels
    L = 1024
    types = ("ring", "disk", "cylshell", "cylinder")
    descs = [kernels.window_desc(t, 0.02 * L * (i + 1), 0.015 * L * i, axis=1) for i, t in enumerate(types)]
    print("line of sight J=10", flush=True)
    _compare(phi, 10, torch.float32, descs, 210)


@pytest.mark.parametrize("spacing", ["linear", "uneven"])
def test_radial_pass_with_many_channels(phi, spacing):
    """1500 radii at L = 256: 47 KB of channel sums beside the staged powers, above the dynamic LDS a kernel gets
    unasked; a subset of the radii through the general kernel."""
    import torch
    from pyhermes_amd import kernels
    J, L = 8, 256
    R = np.linspace(0.01 * L, 0.3 * L, 1500) if spacing == "linear" else np.geomspace(0.01 * L, 0.3 * L, 1500)
    descs = [kernels.window_desc("shell", r) for r in R]
    F1, F2, P, scale = _spectra(phi, J, torch.float64, 11)
    print(f"radial J=8 1500 channels {spacing}", flush=True)
    got = kernels.pair_reduce(F1, F2, P, descs)
    ref = kernels.pair_reduce(F1, F2, P, descs[::75] + [kernels.window_desc("sphere", 2.0)])[:-1]
    assert np.abs(got[::75] - ref).max() <= 1e-12 * scale
