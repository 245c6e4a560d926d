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
    # at most 729 vertices, or 1331 where an axis has an odd number of elements (9 x 10 x 11)
    assert info["level_size"][-1] <= 1331 and info["dense_coarsest"]
    # CG stops at 1e-12 of the preconditioned residual; as in test_gpu_dsa.py
    assert np.linalg.norm(x - ref) < 1e-9 * np.linalg.norm(ref)


def _quarter_turn(v):
    """The axes of the mesh one coordinate on: no axis lies along its own coordinate."""
    return np.ascontiguousarray(np.stack([-v[:, 1], v[:, 0]], 1) if v.shape[1] == 2 else v[:, [2, 0, 1]])


def _half_ring(v):
    r, th = 1.0 + v[:, 1], np.pi * (1.0 - v[:, 0])
    return np.ascontiguousarray(np.stack([r * np.cos(th), r * np.sin(th)], 1))


@pytest.mark.parametrize("nel,ext,turn", [((64, 64), (1.0, 1.0), _quarter_turn), ((24, 24, 24), (1.0, 1.0, 1.0), _quarter_turn),
                                          ((96, 24), (1.0, 2.0), _quarter_turn), ((64, 48), (1.0, 1.0), _half_ring)])
def test_coarsening_follows_the_grid_axes(nel, ext, turn):
    """A mesh whose axes are not coordinate axes coarsens like one with the same edges
    along the coordinates, and needs as many CG iterations."""
    print(f"dsa axes {nel} {turn.__name__}", flush=True)
    ne = int(np.prod(nel))
    rng = np.random.default_rng(3)
    st = P.lognormal_sigma(ne, 1.0, rng) * 5
    b = rng.normal(size=ne * 2 ** len(nel))
    up = P.cartesian_vertices(nel, extents=ext)
    # the ring's mean radius is 1.5: the same edge lengths on a box
    box = P.cartesian_vertices(nel, extents=(1.5 * np.pi, 1.0)) if turn is _half_ring else up
    got = []
    for v in (box, turn(up)):
        op = A.InverseAdvectionOperator(A.Mesh(nel, vertices=v), 1, 4, st)
        dsa = A.DSA(op, 0.99 * st, cg_reltol=1e-8, cg_maxit=200)
        dsa.solve(b)
        got.append(dsa.info())
    print(f"  levels {got[1]['level_size']} CG its {[g['last_cg_iterations'] for g in got]}", flush=True)
    assert got[0]["level_size"] == got[1]["level_size"]
    # a turned box is the same operator; the ring's cells differ by a factor 2 in width
    assert got[1]["last_cg_iterations"] <= got[0]["last_cg_iterations"] + (0 if turn is _quarter_turn else 6)


@pytest.mark.parametrize("nel,its", [((33, 33), 7), ((600, 1), 4), ((9, 10, 9), 8), ((66, 66), 13)])
def test_small_odd_grids_keep_the_dense_inverse(nel, its):
    """A vertex grid of 730 to 1331 vertices that does not halve evenly is the coarsest:
    the vertex space is solved exactly and CG needs no more iterations than that allows."""
    print(f"dsa small odd {nel}", flush=True)
    ne = int(np.prod(nel))
    rng = np.random.default_rng(2)
    st = P.lognormal_sigma(ne, 1.0, rng) * 5
    op = A.InverseAdvectionOperator(A.Mesh(nel), 1, 4, st)
    dsa = A.DSA(op, 0.99 * st, cg_reltol=1e-8, cg_maxit=200)
    dsa.solve(rng.normal(size=op.phi_size))
    info = dsa.info()
    print(f"  levels {info['level_size']} CG its {info['last_cg_iterations']}", flush=True)
    assert 729 < info["level_size"][-1] <= 1331 and info["dense_coarsest"]
    assert info["last_cg_iterations"] <= its + 1
