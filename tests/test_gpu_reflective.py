"""Reflective sides with several groups and an unaligned mesh, every level
kernel against the oracle.  A direction that leaves through a reflective side
has no reflected partner (its table entry is -1), and no kernel may form an
address from that entry: group 0 would read below psi."""
import numpy as np
import pytest

import allium_amd as A
import oracle
from allium_amd import problems as P
from tests.helpers import ls_fixture, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nel,p,jitter", [((11, 36), 1, 0.0), ((7, 9), 2, 0.05), ((5, 4, 6), 1, 0.05),
                                          ((3, 4, 3), 2, 0.0), ((3, 3, 4), 2, 0.05)])
@pytest.mark.parametrize("lanes", [0, 1, 2, 4])
def test_reflective_groups_match_oracle(nel, p, jitter, lanes):
    dim, n = len(nel), (p + 1) ** len(nel)
    if (lanes == 0 and jitter) or (lanes and n % lanes) or (dim == 3 and p == 2 and lanes != 1):
        pytest.skip("no such layout for this element")
    print(f"reflective {nel} p={p} jitter {jitter} lanes {lanes}", flush=True)
    rng = np.random.default_rng(3)
    ne, G = int(np.prod(nel)), 3
    sig = np.stack([P.lognormal_sigma(ne, 1.0, rng) for _ in range(G)])
    v = P.jittered_vertices(nel, jitter, rng) if jitter else P.cartesian_vertices(nel)
    bc = (0, 1) + (0,) * (2 * dim - 2)
    op = A.InverseAdvectionOperator(A.Mesh(nel, vertices=v, bc=bc), p, 4, sig)
    op.set_tuning(0, 64, lanes)
    om, w = ls_fixture(4, dim)
    pr = oracle.Problem(dim, nel, v, p, om, w, sig, bc=bc)
    q = rng.uniform(0.1, 1.0, op.size)
    ref = np.empty(op.size)
    pr.sweep(q, ref)
    psi = A.DeviceVector(op.size)
    op.Mult(A.DeviceVector.from_host(q), psi)
    # 1e-12: both solve the same FP64 cell systems, in other elimination orders
    assert rel_err(psi.to_host(), ref) < 1e-12
