"""Strided passes of the 3-D transforms (grids of 128^3 and more): half spectra, whose rows start anywhere in a cache
line and whose last tile holds one column, and full ones; both precisions and directions; batches; the library plan
below.  Oracle: torch.fft in FP64.  A transform of white noise has white rounding errors: one unit per radix-2 level
in each of them, log2(N) levels, so sqrt(log2 N) eps of the rms; the largest of up to 10^9 errors is about 6.5 sigma
and the oracle's own FP64 error adds as much, so 16 eps sqrt(log2 N) of the rms holds with room."""
import numpy as np
import pytest
import torch

from pyhermes_amd import kernels

pytestmark = pytest.mark.gpu


def _field(shape, dtype, seed=3):
    return torch.randn(shape, generator=torch.Generator(device="cuda").manual_seed(seed), device="cuda", dtype=dtype)


def _check(got, want, J, dtype):
    eps = 2.0 ** (-24 if dtype == torch.float32 else -53)
    rms = float(want.abs().square().mean().sqrt())
    assert float((got.to(want.dtype) - want).abs().max()) <= 16.0 * eps * np.sqrt(3 * J) * rms


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("J,batch", [(6, 1), (7, 1), (7, 3), (8, 1), (9, 1), (10, 1)])
def test_half_spectrum(J, batch, dtype):
    L = 1 << J
    x = _field((batch, L, L, L), dtype)
    spec = kernels.rfftn(x)
    if J < 10:
        _check(spec, torch.fft.rfftn(x.double(), dim=(-3, -2, -1)), J, dtype)
    else:  # the largest grid against its own rows: one plane at a time
        part = torch.fft.rfft(x.double(), dim=-1)[..., 5:6]
        _check(spec[..., 5:6], torch.fft.fft2(part, dim=(-3, -2)), J, dtype)
        del part
    back = kernels.irfftn_unnormalized(spec, L)
    _check(back / float(L) ** 3, x.double(), 2 * J, dtype)


@pytest.mark.parametrize("dtype", [torch.complex64, torch.complex128])
@pytest.mark.parametrize("inverse", [False, True])
@pytest.mark.parametrize("J,batch", [(6, 2), (7, 2), (8, 1), (9, 1)])
def test_full_spectrum(J, batch, inverse, dtype):
    L = 1 << J
    x = _field((batch, L, L, L), dtype)
    fn = torch.fft.ifftn if inverse else torch.fft.fftn
    want = fn(x.to(torch.complex128), dim=(-3, -2, -1), norm="forward" if inverse else "backward")
    real = torch.float32 if dtype == torch.complex64 else torch.float64
    keep = x.clone()
    _check(kernels.fftn_c2c(x, inverse=inverse), want, J, real)
    assert torch.equal(x, keep)
    _check(kernels.fftn_c2c(x, inverse=inverse, out=x), want, J, real)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("J", [6, 7, 8, 9])
def test_convolution(J, dtype):
    """Two transforms and products of O(1): the bound of a transform of twice the levels."""
    L = 1 << J
    x = _field((L, L, L), dtype)
    f = _field((L // 2 + 1,), dtype, 4)  # a product symmetric under k -> -k, as windows are
    full = torch.cat([f, f[1:-1].flip(0)])
    k = full[:, None, None] * full[None, :, None] * f
    keep = x.clone()
    got = kernels.convolve_real(x, k, 1.0 / L ** 3)
    spec = torch.fft.rfftn(x.double())
    spec *= k.double()
    _check(got, torch.fft.irfftn(spec, s=(L, L, L)), 2 * J, dtype)
    assert torch.equal(x, keep)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_convolution_of_the_largest_grid(dtype):
    """L = 1024 (up to 147 KB of LDS in the fused pass), with a product of one filter per axis, so that the reference
    is three passes of 1-D transforms."""
    J = 10
    L = 1 << J
    x = _field((L, L, L), dtype)
    f = _field((L // 2 + 1,), dtype, 4)
    full = torch.cat([f, f[1:-1].flip(0)])
    k = full[:, None, None] * full[None, :, None] * f
    print(f"convolution J=10 {dtype}", flush=True)
    got = kernels.convolve_real(x, k, 1.0 / L ** 3)
    del k
    want = x.double()
    del x
    shape = [(L // 2 + 1, 1, 1), (L // 2 + 1, 1), (L // 2 + 1,)]
    for axis in range(3):
        spec = torch.fft.rfft(want, dim=axis)
        spec *= f.double().view(shape[axis])
        want = torch.fft.irfft(spec, n=L, dim=axis)
        del spec
    _check(got, want, 2 * J, dtype)
