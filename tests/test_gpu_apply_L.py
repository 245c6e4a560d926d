"""The streaming operator on general geometry, whose lanes take the directions of an
element: groups, the time mass, direction counts below, at and off a wave."""
import numpy as np
import pytest

import allium_amd as A
import oracle
from allium_amd import problems as P
from tests.helpers import ls_fixture, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nel,p,sn,G,tau", [((7, 5), 1, 4, 2, 0.0), ((4, 3), 2, 12, 1, 1.5), ((3, 4, 2), 1, 8, 2, 0.7),
                                            ((1, 2, 1), 2, 2, 3, 0.0), ((3, 2, 4), 2, 6, 2, 2.5), ((9, 1), 0, 8, 1, 0.0)])
def test_apply_L_general_geometry(nel, p, sn, G, tau):
    print(f"apply L {nel} p={p} S{sn} G={G} tau {tau}", flush=True)
    rng = np.random.default_rng(8)
    ne = int(np.prod(nel))
    sig = np.stack([P.lognormal_sigma(ne, 1.0, rng) for _ in range(G)])
    v = P.jittered_vertices(nel, 0.05, rng)
    v[0] += 0.01   # general geometry on meshes without interior vertices too
    op = A.InverseAdvectionOperator(A.Mesh(nel, vertices=v), p, sn, sig)
    om, w = ls_fixture(sn, len(nel))
    pr = oracle.Problem(len(nel), nel, v, p, om, w, sig)
    if tau:
        op.SetTimeAbsorption(tau)
        pr.set_time_absorption(tau)
    x = rng.uniform(-1.0, 1.0, op.size)
    # as in test_gpu_sweep.py: sums of up to 27 products per face and element
    assert rel_err(A.AdvectionOperator(op).Mult(x, np.empty_like(x)), pr.apply_L(x)) < 1e-13
