"""The diffusion multigrid on element counts that do not halve evenly: the
solve against a direct one, and a hierarchy that reaches a small grid."""
import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spla

import allium_amd as A
from allium_amd import problems as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nel,p,jitter,smooth", [((41, 36), 1, 0.0, 2), ((53, 29), 2, 0.1, 1), ((900, 1), 1, 0.0, 2),
                                                 ((11, 9, 13), 1, 0.0, 2), ((13, 12, 10), 1, 0.1, 3),
                                                 ((1, 2, 301), 1, 0.0, 2), ((9, 10, 11), 2, 0.0, 1)])
def test_uneven_coarsening_solves(nel, p, jitter, smooth):
    print(f"dsa coarsening {nel} p={p} smooth {smooth}", flush=True)
    dim, ne = len(nel), int(np.prod(nel))
    rng = np.random.default_rng(2)
    vert = P.jittered_vertices(nel, jitter, rng) if jitter else None
    st = P.lognormal_sigma(ne, 1.0, rng) * 5
    op = A.InverseAdvectionOperator(A.Mesh(nel, vertices=vert), p, 4, st)
    # the 1 x 2 x 301 mesh has cells 300 times as wide as thick, where point smoothing gains a
    # digit in about 40 iterations (334 for 8 digits): 12 digits stay below 2000
    dsa = A.DSA(op, 0.99 * st, cg_reltol=1e-12, cg_maxit=2000, smooth=smooth)
    rp, col, val = A.host_mip_matrix(op.mesh, p, 4, st, 0.99 * st)
    K = sp.csr_matrix((val, col, rp), shape=(rp.size - 1,) * 2)
    b = rng.normal(size=K.shape[0])
    x = dsa.solve(b)
    ref = spla.spsolve(sp.csc_matrix(K), b)
    info = dsa.info()
    print(f"  levels {info['level_size']} CG its {info['last_cg_iterations']}", flush=True)
    assert info["level_size"][-1] <= 729 and info["dense_coarsest"]
    # CG stops at 1e-12 of the preconditioned residual; as in test_gpu_dsa.py
    assert np.linalg.norm(x - ref) < 1e-9 * np.linalg.norm(ref)
