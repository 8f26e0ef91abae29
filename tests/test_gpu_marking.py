"""The device marking of the active cones against the host's where its forms change: bitmaps in
LDS and in memory (fine grids of more cells than the LDS copy holds), target boxes larger and
smaller than a workgroup's run of points."""
import numpy as np
import pytest

import ifgf_amd
from conftest import sphere
from test_gpu_tree import _plans_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kappa,n,m,leaf", [
    (4.0, 3000, 3000, 16),     # bitmaps of a few words
    (160.0, 2000, 2000, 40),   # the upper levels' bitmaps exceed the LDS copy
    (8.0, 3000, 30000, 40),    # target boxes of many points
    (8.0, 9000, 700, 64),      # few targets
])
def test_device_marking_matches_host(gpu, kappa, n, m, leaf):
    x = sphere(n, 601)
    y = x if m == n else sphere(m, 602) * 0.2 + np.array([2.5, 0.0, 0.1])
    dev = ifgf_amd.HelmholtzIfgfOperator(kappa, leaf, 6, 1, -1)
    dev.init(x.T, y.T)
    host = ifgf_amd.HelmholtzIfgfOperator(kappa, leaf, 6, 1, -1)
    host.init(x.T, y.T, host_plan=True)
    assert dev.plan_counts()["far_pairs"] > 0
    _plans_equal(dev, host)
