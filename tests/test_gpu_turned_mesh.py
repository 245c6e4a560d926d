"""A box grid turned by 180 degrees about one axis: the coordinates fall along the
logical axes, so the low side of an element is not the one with the smaller
coordinate, and the kernels of upright uniform boxes must not take it."""
import numpy as np
import pytest

import allium_amd as A
import oracle
from allium_amd import problems as P
from tests.helpers import ls_fixture, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nel,p", [((6, 5), 1), ((4, 7), 2), ((3, 4, 5), 1), ((3, 2, 3), 2)])
def test_turned_grid_matches_oracle(nel, p):
    print(f"turned {nel} p={p}", flush=True)
    dim, ne = len(nel), int(np.prod(nel))
    v = P.cartesian_vertices(nel, extents=(1.0, 2.0, 1.5)[:dim])
    v[:, :2] *= -1.0
    sig = P.lognormal_sigma(ne, 1.0, np.random.default_rng(1)).reshape(1, -1)
    op = A.InverseAdvectionOperator(A.Mesh(nel, vertices=v), p, 4, sig)
    om, w = ls_fixture(4, dim)
    pr = oracle.Problem(dim, nel, v, p, om, w, sig)
    q = np.random.default_rng(2).uniform(0.1, 1.0, op.size)
    ref = np.empty(op.size)
    pr.sweep(q, ref)
    dq, psi = A.DeviceVector.from_host(q), A.DeviceVector(op.size)
    for mode in (0, 1) if (dim, p) == (3, 2) else (0, 1, 3):
        op.set_launch(mode)
        psi.upload(np.full(op.size, np.nan))
        op.Mult(dq, psi)
        # 1e-12: both solve the same FP64 cell systems, in other elimination orders
        assert rel_err(psi.to_host(), ref) < 1e-12, mode
