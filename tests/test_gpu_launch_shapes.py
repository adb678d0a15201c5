"""Sizes at which a kernel's launch shape could go wrong: remainders of waves,
blocks and tiles, the smallest sizes and the first past a boundary."""
import numpy as np
import pytest

from fastipc_amd import _lib

pytestmark = pytest.mark.gpu

NPTS = (2, 3, 4, 4, 4, 4, 4)


def _constraints(kind, X, X0, project=1):
    n, nd = len(X), 3 * NPTS[kind]
    E, g, H = np.zeros(n), np.zeros((n, nd)), np.zeros((n, nd, nd))
    _lib.call("fipc_batch_constraint", kind, n, _lib.dptr(X), _lib.dptr(X0), 1e-2, 1.0, project, _lib.dptr(E),
              _lib.dptr(g), _lib.dptr(H))
    return E, g, H


@pytest.mark.parametrize("kind", range(7))
def test_contact_rows_do_not_depend_on_their_number(kind):
    """A row's gradient and projected Hessian are the same bits whether it is
    alone, in a partial group of lanes, or in the last block (4 or 8 rows per
    wave, 16 or 32 per block of the projection)."""
    rng = np.random.default_rng(kind)
    X = np.ascontiguousarray(rng.normal(0, 0.03, (70, NPTS[kind], 3)))
    if kind >= 4:  # nearly parallel edges, so that the mollifier acts
        X[:, 3] = X[:, 2] + (X[:, 1] - X[:, 0]) + rng.normal(0, 1e-3, (70, 3))
    X0 = np.ascontiguousarray(X + rng.normal(0, 0.01, X.shape))
    whole = _constraints(kind, X, X0)
    # projected: positive semi-definite up to the projection's rounding
    for H in whole[2]:
        assert np.linalg.eigvalsh(H)[0] >= -1e-9 * max(np.abs(H).max(), 1e-300)
    for n in (1, 3, 4, 5, 8, 9, 16, 17, 33, 64, 65):
        part = _constraints(kind, X[:n].copy(), X0[:n].copy())
        for a, b in zip(part, whole):
            assert np.array_equal(a, b[:n], equal_nan=True), n
