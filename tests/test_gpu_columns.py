"""Several density columns in one pass against the same columns one by one, where the kernels of
columns.hip change form: numbers of columns at the edges of the groups of up to five columns, of
the 16-wide column tiles and of the register instances, few and many fine coefficients (source boxes per step, products too large
for LDS), fine factor 1, targets other than the sources, passes of unequal width."""
import os

import numpy as np
import pytest

import ifgf_amd
from conftest import cdens, sphere, spheroid

pytestmark = pytest.mark.gpu

# both forms sum the same terms in another order: rounding of some hundred terms
TOL = {"fp64": 1e-12, "mixed": 3e-6}


def _check(op, W, prec):
    U = op.mult(W)
    os.environ["IFGF_NO_BATCH"] = "1"
    try:
        ref = op.mult(W)
    finally:
        del os.environ["IFGF_NO_BATCH"]
    for c in range(W.shape[1]):
        d = np.linalg.norm(U[:, c] - ref[:, c]) / np.linalg.norm(ref[:, c])
        assert d < TOL[prec], (c, d)


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("ncol", [3, 4, 5, 6, 7, 8, 9, 11, 12, 13, 16, 17, 25, 32, 33])
def test_numbers_of_columns(gpu, ncol, prec):
    x, y = spheroid(3000, 81), sphere(1111, 82) * 1.5
    W = np.stack([cdens(3000, 200 + c) for c in range(ncol)], axis=1)
    op = ifgf_amd.HelmholtzIfgfOperator(9.0, 30, 6, 1, -1, precision=prec)
    op.init(x.T, x.T if ncol % 2 else y.T)
    _check(op, W, prec)


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("kind,order,n", [
    ("laplace", 7, 2500),       # 16 coefficients, one radial
    ("laplace", 8, 2500),       # 50: three source boxes per step
    ("laplace", 9, 2500),       # 108: one
    ("laplace", 11, 1500),      # 320
    ("modhelmholtz", 13, 900),  # 700, no compiled first order, fine factor 1
    ("modhelmholtz", 8, 2500),
])
@pytest.mark.parametrize("ncol", [6, 13])  # far field by groups of columns, by 16-wide tiles
def test_orders_of_columns(gpu, kind, order, n, prec, ncol):
    x = spheroid(n, 83)
    if kind == "laplace":
        op = ifgf_amd.LaplaceIfgfOperator(20, order, 1, -1, precision=prec)
        W = np.stack([cdens(n, 300 + c).real for c in range(ncol)], axis=1)
    else:
        op = ifgf_amd.MofifiedHelmholtzIfgfOperator(0.5 - 6.0j, 20, order, 1, -1, precision=prec)
        W = np.stack([cdens(n, 300 + c) for c in range(ncol)], axis=1)
    op.init(x.T, x.T)
    _check(op, W, prec)


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("ncol", [3, 13])
@pytest.mark.parametrize("kind", ["helmholtz", "laplace", "grad"])
def test_densities_that_are_not_finite(gpu, kind, ncol, prec):
    """A density that is not finite leaves the result at its own point, which the sum leaves out,
    as finite as a single column does, and the other columns alone."""
    n = 2000
    x = spheroid(n, 84)
    op = {"helmholtz": lambda: ifgf_amd.HelmholtzIfgfOperator(7.0, 20, 7, 1, -1, precision=prec),
          "laplace": lambda: ifgf_amd.LaplaceIfgfOperator(20, 7, 1, -1, precision=prec),
          "grad": lambda: ifgf_amd.GradHelmholtzIfgfOperator(0.5 - 6.0j, 20, 8, 1, -1,
                                                             precision=prec)}[kind]()
    if kind == "grad":
        op.setDx(0)
    op.init(x.T, x.T)
    W = np.stack([cdens(n, 500 + c) for c in range(ncol)], axis=1)
    W = W.real.copy() if kind == "laplace" else W
    good = op.mult(W)
    W[5, 0], W[6, 1] = np.nan, np.inf
    U = op.mult(W)
    assert np.array_equal(U[:, 2:], good[:, 2:])
    for c in (0, 1):
        u = op.mult(np.ascontiguousarray(W[:, c]))
        assert np.array_equal(np.isfinite(U[:, c]), np.isfinite(u)) and np.isfinite(u).any()
