"""The FP64 triple-product contraction on grids of every size class and for any 3 x 3 overlap matrix.

Tolerance: FP64 sums of L^3 terms whose magnitudes add up to `scale`, a few dozen roundings deep: 1e-13 of it."""

import numpy as np
import pytest

from oracle import multipole as om

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L", [4, 8, 32, 64, 128])
def test_summand_any_overlap_matrix(L):
    import torch
    from pyhermes_amd import kernels
    rng = np.random.default_rng(L)
    d = rng.normal(size=(L, L, L))
    F = [rng.normal(size=(L, L, L)) + 1j * rng.normal(size=(L, L, L)) for _ in range(2)]
    g = rng.normal(size=(3, 3))  # not symmetric
    got = kernels.multipole_summand_f64(kernels.as_device(d, torch.float64), kernels.as_device(F[0], torch.complex128),
                                        kernels.as_device(F[1], torch.complex128), g)
    ref = om.summand_c(d, F[0], F[1], g)
    scale = np.abs(g).sum() ** 3 * np.sqrt((d ** 2).sum() * (np.abs(F[0]) ** 2).mean() * (np.abs(F[1]) ** 2).sum())
    assert abs(got - ref) <= 1e-13 * scale, (got, ref, scale)


def test_plain_multipoles_of_fields_in_another_memory_order(phi):
    """Fields given as permuted views: the multipoles of the same values laid out in order.  The sums differ by the
    roundings of transforms and contractions that see the same numbers: none."""
    import torch
    from pyhermes_amd import kernels, multipole
    L = 16
    geo = multipole.MultipoleGeometry(phi, L)
    rng = np.random.default_rng(2)
    d = [kernels.as_device(rng.normal(size=(L, L, L)), torch.float64).permute(p) for p in ((2, 0, 1), (0, 2, 1), (1, 2, 0))]
    assert not any(t.is_contiguous() for t in d)
    got = multipole.ddd_multipole_plain_f64(geo, *d, 2.5, 4.0, 0, 2)
    want = multipole.ddd_multipole_plain_f64(geo, *(t.contiguous() for t in d), 2.5, 4.0, 0, 2)
    assert np.array_equal(np.asarray(got), np.asarray(want))
