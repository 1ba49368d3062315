"""The octant builders: windows evaluated once per octant position and mirrored, and the fused product.

Against the oracle's own builders at every position; the tolerance is the FP64 rounding of eight alias terms
(each below a few ulps of max |K| after argument errors 2 pi k R 2^-53 < 1e-14): 1e-12 of max |K|."""

import numpy as np
import pytest

from oracle import radial, scaling, windows as ow

pytestmark = pytest.mark.gpu


def _P(phi, L):
    import torch
    from pyhermes_amd import kernels
    P = scaling.fourier_power_spectrum(phi, 0, 1, L, 1024)
    return P, kernels.as_device(P, torch.float64)


@pytest.mark.parametrize("J", [2, 4])
@pytest.mark.parametrize("l,m", [(0, 0), (1, -1), (2, 0), (3, 2), (5, -4), (7, 7), (10, 3)])
@pytest.mark.parametrize("R", [0.01, 2.3, 11.0])
def test_multipole_builder_and_product(phi, J, l, m, R):
    import torch
    from pyhermes_amd import kernels
    L = 1 << J
    P, Pd = _P(phi, L)
    ref = ow.radial_multipole_window(L, P, R, l, m)
    tol = 1e-12 * max(np.abs(ref).max(), 1e-300)
    got = kernels.window_build_full(J, Pd, kernels.window_desc("shell_multipole", R, l=l, m=m)).cpu().numpy()
    assert np.abs(got - ref).max() <= tol
    rng = np.random.default_rng(l)
    spec = rng.normal(size=(L, L, L)) + 1j * rng.normal(size=(L, L, L))
    sd = kernels.as_device(spec, torch.complex128)
    out = kernels.window_apply_full_f64(sd, Pd, kernels.radial_profile("shell", R), l, m, 0.25, torch.empty_like(sd))
    assert np.abs(out.cpu().numpy() - 0.25 * spec * ref).max() <= tol * np.abs(spec).max()


@pytest.mark.parametrize("J", [1, 3, 5])
@pytest.mark.parametrize("wt,a0,a1", [("sphere", 1.7, 0.0), ("gaussian", 0.8, 0.0), ("thick_shell", 3.0, 1.0),
                                      ("gaussian_shell", 2.0, 0.7), ("shell", 4.4, 0.0), ("inverse_laplacian", 0.0, 0.0)])
def test_full_builder_of_real_windows_extends_the_half_grid_one(phi, J, wt, a0, a1):
    """The complex full-grid kernel of a real window repeats its rFFT-layout kernel at (-x, -y, -z)."""
    from pyhermes_amd import kernels
    L = 1 << J
    _, Pd = _P(phi, L)
    d = kernels.window_desc(wt, a0, a1)
    half = kernels.window_build_rfft(J, Pd, d).cpu().numpy()
    full = kernels.window_build_full(J, Pd, d).cpu().numpy()
    i = (-np.arange(L)) % L
    want = np.empty((L, L, L))
    want[:, :, :L // 2 + 1] = half
    want[:, :, L // 2 + 1:] = half[i][:, i][:, :, 1:L // 2][:, :, ::-1]
    # the two builders add the eight aliases in different orders
    assert np.abs(full.real - want).max() <= 1e-14 * np.abs(want).max()
    assert not full.imag.any()
