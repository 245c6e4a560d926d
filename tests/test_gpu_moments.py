"""The moment kernel on both sides of its size rule, at entry counts around its
64- and 128-entry workgroups and direction counts below and above its waves."""
import numpy as np
import pytest

import allium_amd as A

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nel,p,sn,G", [((1, 1), 0, 2, 1), ((9, 7), 0, 2, 3), ((8, 8), 0, 4, 1), ((16, 1), 1, 2, 2),
                                        ((5, 13), 0, 8, 1), ((11, 6), 2, 12, 2), ((3, 5, 7), 1, 16, 1),
                                        ((47, 50, 49), 1, 8, 1)])
def test_moments_match_the_sum(nel, p, sn, G):
    print(f"moments {nel} p={p} S{sn} G={G}", flush=True)
    ne = int(np.prod(nel))
    op = A.InverseAdvectionOperator(A.Mesh(nel), p, sn, np.ones((G, ne)))
    w = op.quadrature()[1]
    rng = np.random.default_rng(1)
    psi = rng.uniform(-1.0, 1.0, op.size)
    phi = A.DiscreteToMoment(op).Mult(A.DeviceVector.from_host(psi), A.DeviceVector(op.phi_size)).to_host()
    ps = psi.reshape(G, op.Nomega, -1)
    ref = np.einsum("a,gai->gi", w, ps).reshape(-1)
    # each partial sum is rounded once per direction and once per wave
    bound = (op.Nomega + 16) * 2.0 ** -52 * np.einsum("a,gai->gi", w, np.abs(ps)).reshape(-1)
    assert (np.abs(phi - ref) <= bound).all()


@pytest.mark.parametrize("nel,p,sn,G", [((121, 61, 72), 0, 2, 1),       # few directions, many entries
                                        ((263, 251), 0, 4, 9),          # and several groups, rows off 64 bytes
                                        ((13, 7), 0, 4, 2),             # few directions, few entries
                                        ((81, 83, 79), 0, 4, 1),        # 24 directions, rows off 64 bytes
                                        ((5, 5, 5), 0, 6, 4),           # the same with few entries
                                        ((17, 9, 5), 1, 6, 2),          # 12 directions per wave: a chunk of 8 and one of 4
                                        ((58, 59, 58), 1, 8, 1)])       # over 1 GB
def test_moments_of_every_split(nel, p, sn, G):
    test_moments_match_the_sum(nel, p, sn, G)
