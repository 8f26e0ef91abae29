"""The far field with the pair records laid down at init and without them (the targets located in
every mult): the same results, bit for bit, for every form that takes either: single columns at
compiled and other orders, fine factors 1 and 3, several waves per item and one, angle tables in
LDS and too large for it, groups of columns and 16-wide tiles, both precisions, merged operators,
level storage, adjoints of other targets."""
import numpy as np
import pytest

import ifgf_amd
from conftest import cdens, sphere, spheroid

pytestmark = pytest.mark.gpu


def _pair(make, x, y, **kw):
    """(operator with records, without)"""
    ops = []
    for records in (True, False):
        op = make()
        op.init(x.T, y.T, pair_records=records, **kw)
        ops.append(op)
    a, b = (op.plan_counts() for op in ops)
    assert a["far_pairs"] > 0 and b["device_bytes"] < a["device_bytes"]
    return ops


def _same(a, b, w):
    u, v = a.mult(w), b.mult(w)
    assert np.array_equal(u, v), np.linalg.norm(u - v) / np.linalg.norm(u)


def _columns(n, ncol):
    return np.stack([cdens(n, 400 + c) for c in range(ncol)], axis=1)


ORDERS = [
    ("helmholtz", 6, -1.0, 3000, 9.0),        # (3,6,6)/(2,3,3)
    ("helmholtz", 8, -1.0, 3000, 9.0),        # (5,8,8)/(2,5,5)
    ("helmholtz", 6, 1e-5, 12000, 16.0),      # (6,8,7)/(3,5,4)
    ("helmholtz", 3, -1.0, 2500, 7.0),        # (2,3,3)/(2,2,2)
    ("helmholtz", 7, -1.0, 2500, 7.0),        # (4,7,7)/(2,4,4)
    ("laplace", 7, -1.0, 2500, 0.0),          # one radial coefficient
    ("laplace", 10, -1.0, 2500, 0.0),         # (7,10,10)/(4,7,7)
    ("laplace", 12, -1.0, 1500, 0.0),         # (9,12,12)/(6,9,9)
    ("modhelmholtz", 8, -1.0, 2500, 6.0),     # fine factor 1
    ("modhelmholtz", 13, -1.0, 900, 6.0),     # no compiled first order
    ("helmholtz", 6, -1.0, 1500, 700.0),      # angle tables too large for LDS
]


def _make(kind, order, tol, k, prec):
    leaf = 64 if tol > 0 else 20
    if kind == "laplace":
        return lambda: ifgf_amd.LaplaceIfgfOperator(leaf, order, 1, tol, precision=prec)
    if kind == "modhelmholtz":
        return lambda: ifgf_amd.MofifiedHelmholtzIfgfOperator(0.5 - 1j * k, leaf, order, 1, tol,
                                                              precision=prec)
    return lambda: ifgf_amd.HelmholtzIfgfOperator(k, leaf, order, 1, tol, precision=prec)


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("kind,order,tol,n,k", ORDERS)
def test_orders_and_columns(gpu, kind, order, tol, n, k, prec):
    x = spheroid(n, 501) if tol < 0 else sphere(n, 100 + n % 97)
    a, b = _pair(_make(kind, order, tol, k, prec), x, x)
    for ncol in (1, 4, 5, 12, 13, 32):
        print(f"{kind} order {order} prec={prec} columns={ncol}", flush=True)
        W = _columns(n, ncol)
        _same(a, b, W.real.copy() if kind == "laplace" else W)


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("order,tol", [(6, -1.0), (7, -1.0), (6, 1e-4)])
def test_one_wave_per_item(gpu, order, tol, prec):
    """Launches of more items than are split over waves, workgroups of several items."""
    x = sphere(600000, 504)
    a, b = _pair(lambda: ifgf_amd.HelmholtzIfgfOperator(40.0, 64, order, 1, tol, precision=prec),
                 x, x)
    w = cdens(600000, 505)
    for waves in (1, 2, 8):
        a.launch_shape = b.launch_shape = dict(far_waves=waves)
        _same(a, b, w)


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_other_targets_adjoint_level_storage_and_merged(gpu, prec, tmp_path):
    x, y = spheroid(4000, 506), sphere(2500, 507) * 1.4
    make = lambda: ifgf_amd.HelmholtzIfgfOperator(9.0, 30, 6, 1, -1, precision=prec)
    a, b = _pair(make, x, y)
    for ncol in (1, 5, 16):
        _same(a, b, _columns(4000, ncol))
        g = _columns(2500, ncol)
        assert np.array_equal(a.mult_adjoint(g), b.mult_adjoint(g))
    ra, rb = _pair(make, x, y, level_ring=True)
    _same(ra, rb, cdens(4000, 508))
    a.save_plan(tmp_path / "r.plan")
    c = make()
    c.load_plan(tmp_path / "r.plan", pair_records=False)
    assert c.plan_counts()["device_bytes"] == b.plan_counts()["device_bytes"]
    _same(a, c, cdens(4000, 508))
    parts = []
    for i, k in enumerate((5.0, 12.0)):
        op = ifgf_amd.HelmholtzIfgfOperator(k, 30, 6, 1, -1, precision=prec)
        p = sphere(3000 - 1000 * i, 510 + i)
        op.init(p.T, p.T)
        parts.append(op)
    ma, mb = ifgf_amd.merge(parts), ifgf_amd.merge(parts, pair_records=False)
    assert mb.plan_counts()["device_bytes"] < ma.plan_counts()["device_bytes"]
    for ncol in (1, 4, 14):
        _same(ma, mb, _columns(5000, ncol))


def test_records_leave_the_margin_free(gpu):
    """With 4 GiB and twice the records' memory left an operator goes without records (they take at
    most a quarter of what there is beyond 4 GiB); with the memory given back it has them."""
    import torch
    GiB = 1 << 30
    x, w = sphere(60000, 520), cdens(60000, 521)
    make = lambda: ifgf_amd.HelmholtzIfgfOperator(20.0, 64, 6, 1, -1)
    a, b = _pair(make, x, x)
    u = a.mult(w)
    have, bare = (op.plan_counts()["device_bytes"] for op in (a, b))
    rec = have - bare
    print(f"pair records {rec / GiB:.2f} GiB", flush=True)
    assert GiB // 4 < rec < 2 * GiB
    del a, b
    torch.cuda.empty_cache()
    left = bare + 4 * GiB + 2 * rec
    filler = torch.empty(torch.cuda.mem_get_info()[0] - left, dtype=torch.uint8, device="cuda:0")
    op = make()
    op.init(x.T, x.T)
    c = op.plan_counts()
    assert c["device_bytes"] == bare and c["level_ring"] == 0
    assert np.array_equal(op.mult(w), u)
    del filler
    torch.cuda.empty_cache()
    op.init(x.T, x.T)
    assert op.plan_counts()["device_bytes"] == have and np.array_equal(op.mult(w), u)
