"""The fused window kernel with its shells split over workgroups (small grids) equals one shell at a time.

Each shell's field is computed by the same instructions whatever the group it falls in: bit for bit."""

import numpy as np
import pytest

from oracle import scaling

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("J,n_shell", [(3, 5), (5, 16), (6, 1), (6, 7), (6, 16), (7, 3), (8, 3)])
def test_shell_groups(phi, J, n_shell):
    import torch
    from pyhermes_amd import kernels
    L = 1 << J
    P = kernels.as_device(scaling.fourier_power_spectrum(phi, 0, 1, L, 1024), torch.float64)
    gen = torch.Generator(device="cuda").manual_seed(J)
    H = kernels.rfftn(torch.randn((L, L, L), generator=gen, device="cuda"))
    radii = np.linspace(0.05, 0.3, n_shell) * L
    out = torch.empty((2 * n_shell, L, L, L), dtype=torch.complex64, device="cuda")
    kernels.multipole_window_ifft_multi_f32(H, P, radii, 4, [1, 3], 1.0, out)
    packed = torch.empty((n_shell, L, L, L), dtype=torch.complex64, device="cuda")
    kernels.multipole_window_ifft_pack0_f32(H, P, radii, 2, 1.0, packed)
    one = torch.empty((2, L, L, L), dtype=torch.complex64, device="cuda")
    for s in range(n_shell):
        kernels.multipole_window_ifft_multi_f32(H, P, radii[s:s + 1], 4, [1, 3], 1.0, one)
        assert torch.equal(out[s], one[0]) and torch.equal(out[n_shell + s], one[1])
        kernels.multipole_window_ifft_pack0_f32(H, P, radii[s:s + 1], 2, 1.0, one[:1])
        assert torch.equal(packed[s], one[0])
