"""Operators at orders without a compiled order class, against the oracle: the kernels that take
the orders at run time, at the edges of their first-order and second-order instances, of the
coefficient chunks and of the LDS forms."""
import numpy as np
import pytest

import ifgf_amd
from conftest import cdens, sphere, spheroid
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


def _op(kind, k, leaf, order, prec):
    if kind == po.LAPLACE:
        return ifgf_amd.LaplaceIfgfOperator(leaf, order, 1, -1, precision=prec)
    if kind == po.MODHELMHOLTZ:
        return ifgf_amd.MofifiedHelmholtzIfgfOperator(k, leaf, order, 1, -1, precision=prec)
    return ifgf_amd.HelmholtzIfgfOperator(k, leaf, order, 1, -1, precision=prec)


# FP64 differs from the oracle by rounding only; the mixed form by FP32 rounding of sums of
# some hundred terms (about 1e-7 relative each, partly adding up)
TOL = {"fp64": 1e-11, "mixed": 5e-6}


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("kind,k,order,n", [
    (po.HELMHOLTZ, 7.0, 3, 2500),             # (2,3,3)/(2,2,2): the smallest orders
    (po.HELMHOLTZ, 7.0, 5, 2500),             # (2,5,5)/(2,2,2)
    (po.HELMHOLTZ, 7.0, 7, 2500),             # (4,7,7)/(2,4,4)
    (po.LAPLACE, 0.0, 7, 2500),               # (4,7,7)/(1,4,4): one radial coefficient
    (po.LAPLACE, 0.0, 9, 2500),               # (6,9,9)/(3,6,6): a plane larger than a chunk
    (po.LAPLACE, 0.0, 10, 2500),              # (7,10,10)/(4,7,7)
    (po.LAPLACE, 0.0, 12, 1500),              # (9,12,12)/(6,9,9): children one after another
    (po.MODHELMHOLTZ, 0.5 - 6.0j, 13, 900),   # (10,13,13)/(7,10,10): no compiled first order
    (po.MODHELMHOLTZ, 0.5 - 6.0j, 8, 2500),   # (5,8,8)/(2,5,5), fine factor 1
    (po.MODHELMHOLTZ, 0.5 - 6.0j, 11, 1500),  # (8,11,11)/(5,8,8), fine factor 1
])
def test_orders_against_oracle(gpu, kind, k, order, n, prec):
    x = spheroid(n, 71)
    w = cdens(n, 72)
    if kind == po.LAPLACE:
        w = w.real.copy()
    ref = po.Oracle(kind, k, 20, order, 1, -1.0).init(x, x).mult(w.astype(complex))
    op = _op(kind, k, 20, order, prec)
    op.init(x.T, x.T)
    assert op.plan_counts()["far_pairs"] > 0 and op.plan_counts()["up_table_levels"] > 0
    u = op.mult(w)
    ref = ref.real if kind == po.LAPLACE else ref
    assert np.linalg.norm(u - ref) < TOL[prec] * np.linalg.norm(ref)
