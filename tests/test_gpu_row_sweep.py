"""2D direction sweeps by rows of elements against the oracle: one row, one
column, rows around the 64-lane workgroup and several strips, groups, the time
mass, an isotropic source alone, in place, and unequal element sides."""
import numpy as np
import pytest

import allium_amd as A
import oracle
from allium_amd import problems as P
from tests.helpers import ls_fixture, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p", [1, 2])
@pytest.mark.parametrize("nel,block,G,tau", [((1, 1), 64, 1, 0.0), ((9, 1), 64, 2, 0.0), ((1, 70), 64, 1, 0.0),
                                             ((5, 63), 64, 1, 1.5), ((4, 64), 256, 1, 0.0), ((7, 65), 64, 3, 0.0),
                                             ((3, 200), 64, 1, 0.0), ((33, 130), 128, 2, 0.7), ((66, 40), 512, 1, 0.0)])
def test_rows_match_oracle(nel, p, block, G, tau):
    print(f"rows {nel} p={p} block {block} G={G} tau {tau}", flush=True)
    rng = np.random.default_rng(6)
    ne = int(np.prod(nel))
    sig = np.stack([P.lognormal_sigma(ne, 1.0, rng) for _ in range(G)])
    v = P.cartesian_vertices(nel, extents=(1.0, 3.0))
    op = A.InverseAdvectionOperator(A.Mesh(nel, vertices=v), p, 6, sig)
    op.set_tuning(3, block, 1)
    om, w = ls_fixture(6, 2)
    pr = oracle.Problem(2, nel, v, p, om, w, sig)
    if tau:
        op.SetTimeAbsorption(tau)
        pr.set_time_absorption(tau)
    q = rng.uniform(0.1, 1.0, op.size)
    ref = np.empty(op.size)
    pr.sweep(q, ref)
    # psi starts as NaN: no value of an unsolved cell may reach a result
    psi = A.DeviceVector.from_host(np.full(op.size, np.nan))
    op.Mult(A.DeviceVector.from_host(q), psi)
    # FP64 both; the eigenvectors' condition (7 per axis at p = 2) times rounding stays below
    assert rel_err(psi.to_host(), ref) < 1e-12
    inp = A.DeviceVector.from_host(q)
    op.Mult(inp, inp)
    np.testing.assert_array_equal(inp.to_host(), psi.to_host())
    iso = rng.uniform(0.1, 1.0, (G, 1, ne * (p + 1) ** 2))
    pr.sweep(np.ascontiguousarray(np.broadcast_to(iso, (G, op.Nomega, iso.shape[2]))).reshape(-1), ref)
    phi = A.DeviceVector(op.phi_size)
    op.MultMoments(None, psi, phi, A.DeviceVector.from_host(iso))
    assert rel_err(psi.to_host(), ref) < 1e-12
