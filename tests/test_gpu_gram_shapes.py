"""The Gram contractions at the edges of their tiles and segments, against the FP64 contraction of the oracle.

Tolerance: FP32 products of filtered fields (a few 2^-24 relative, some ten operations deep), summed in FP64 after
at most six planes: 2e-6 of the Cauchy-Schwarz scale, as for the existing sizes."""

import numpy as np
import pytest

from oracle import multipole as om, scaling

pytestmark = pytest.mark.gpu


def _fields(L, n, seed):
    rng = np.random.default_rng(seed)
    return (rng.normal(size=(n, L, L, L)) + 1j * rng.normal(size=(n, L, L, L))).astype(np.complex64)


def _check(d, U, V, g, got, pairs, conj):
    L = d.shape[0]
    for i, j in pairs:
        W = np.conj(V[j]) if conj else V[j]
        a, b = U[i].astype(np.complex128), W.astype(np.complex128)
        ref = om.summand_c(d, a, b, g).real
        scale = np.sqrt(np.sum(d ** 2) * np.sum(np.abs(a) ** 2) * np.sum(np.abs(b) ** 2) / L ** 3)
        assert abs(got[i, j] - ref) <= 2e-6 * scale, (i, j, got[i, j], ref)


@pytest.mark.parametrize("L,n_u,n_v,v_conj,layout", [(8, 3, 2, False, "xmajor"), (8, 16, 16, True, "ymajor"),
                                                    (16, 1, 16, False, "ymajor"), (32, 16, 1, True, "xmajor"),
                                                    (64, 11, 15, False, "ymajor")])
def test_cross_gram(phi, L, n_u, n_v, v_conj, layout):
    from pyhermes_amd import kernels
    import torch
    g = scaling.cal_gamma(phi, 3, 1024)
    lam, Q = np.linalg.eigh(g)
    d = np.random.default_rng(L).normal(size=(L, L, L)).astype(np.float32).astype(np.float64)
    U, V = _fields(L, n_u, 1), _fields(L, n_v, 2)
    order = (lambda a: np.ascontiguousarray(np.swapaxes(a, 1, 2))) if layout == "ymajor" else (lambda a: a)
    with kernels.field_layout(layout):
        got = kernels.multipole_gram_f32(kernels.as_device(d, torch.float32), kernels.as_device(order(U), torch.complex64),
                                         Q, lam, V=kernels.as_device(order(V), torch.complex64), v_conj=v_conj)
    assert got.shape == (n_u, n_v)
    _check(d, U, V, g, got, {(0, 0), (n_u - 1, n_v - 1), (n_u // 2, n_v - 1)}, v_conj)


@pytest.mark.parametrize("nneg", [0, 1, 2, 3])
def test_cross_gram_for_any_eigenvalue_signs(nneg):
    from pyhermes_amd import kernels
    import torch
    L = 16
    rng = np.random.default_rng(nneg)
    Q, _ = np.linalg.qr(rng.normal(size=(3, 3)))
    lam = np.array([0.7, 1.1, 0.4]) * np.where(np.arange(3) < nneg, -1.0, 1.0)
    g = Q @ np.diag(lam) @ Q.T
    d = rng.normal(size=(L, L, L)).astype(np.float32).astype(np.float64)
    U, V = _fields(L, 2, 3), _fields(L, 3, 4)
    got = kernels.multipole_gram_f32(kernels.as_device(d, torch.float32), kernels.as_device(U, torch.complex64), Q, lam,
                                     V=kernels.as_device(V, torch.complex64))
    _check(d, U, V, g, got, {(0, 0), (1, 2)}, False)


@pytest.mark.parametrize("L", [16, 32, 64, 128])
def test_auto_gram_segments(phi, L):
    """Short x segments (8 and 16 planes) where whole columns leave the chip idle."""
    from pyhermes_amd import kernels
    import torch
    g = scaling.cal_gamma(phi, 3, 1024)
    lam, Q = np.linalg.eigh(g)
    d = np.random.default_rng(L).normal(size=(L, L, L)).astype(np.float32).astype(np.float64)
    U = _fields(L, 3, 5)
    got = kernels.multipole_gram_f32(kernels.as_device(d, torch.float32), kernels.as_device(U, torch.complex64), Q, lam)
    _check(d, U, U, g, got, {(0, 0), (1, 2)}, True)
