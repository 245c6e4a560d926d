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


def _extended_sweep(nel, p, om, sigma, q):
    """psi of a unit square box grid in extended precision: LU cell solves along the
    wavefronts, all directions at once.  q and the result: (directions, elements, nodes)."""
    T = np.longdouble
    nx, ny = nel
    m, c = {1: (np.array([[2, 1], [1, 2]], T) / 6, np.array([[1, 1], [-1, 1]], T) / 2),
            2: (np.array([[4, 2, -1], [2, 16, 2], [-1, 2, 4]], T) / 30,
                np.array([[3, 4, -1], [-4, 0, 4], [1, -4, 3]], T) / 6)}[p]
    n, nq = p + 1, (p + 1) ** 2
    hx, hy = T(1) / nx, T(1) / ny
    ax, ay = np.abs(om[:, 0]).astype(T), np.abs(om[:, 1]).astype(T)
    K = ax[:, None, None] * hy * np.kron(m, c) + ay[:, None, None] * hx * np.kron(c, m)
    Mu = hx * hy * np.kron(m, m)
    no = len(om)
    node = np.arange(nq).reshape(n, n)
    psi = np.zeros((no, ny, nx, nq), T)
    qq = q.reshape(no, ny, nx, nq).astype(T)
    sg = np.broadcast_to(sigma.reshape(1, ny, nx), (no, ny, nx)).astype(T)
    flips = []
    for a in range(no):   # every direction swept towards +x, +y in its own orientation
        fx, fy = om[a, 0] < 0, om[a, 1] < 0
        idx = node[::-1] if fy else node
        idx = (idx[:, ::-1] if fx else idx).reshape(-1)
        flips.append((slice(None, None, -1 if fy else 1), slice(None, None, -1 if fx else 1), idx))
    qq = np.stack([qq[a][f[0], f[1]][..., f[2]] for a, f in enumerate(flips)])
    sg = np.stack([sg[a][f[0], f[1]] for a, f in enumerate(flips)])
    for l in range(nx + ny - 1):
        j = np.arange(max(0, l - nx + 1), min(ny, l + 1))
        i = l - j
        A = K[:, None] + sg[:, j, i][..., None, None] * Mu
        x = qq[:, j, i].copy()
        up = np.where((i > 0)[None, :, None], psi[:, j, np.maximum(i - 1, 0)][..., node[:, -1]], T(0))
        x[..., node[:, 0]] += (ax * hy)[:, None, None] * (up @ m)
        up = np.where((j > 0)[None, :, None], psi[:, np.maximum(j - 1, 0), i][..., node[-1]], T(0))
        x[..., node[0]] += (ay * hx)[:, None, None] * (up @ m)
        for k in range(nq):
            f = A[..., k + 1:, k] / A[..., k, k][..., None]
            A[..., k + 1:, k + 1:] -= f[..., None] * A[..., k, k + 1:][..., None, :]
            x[..., k + 1:] -= f * x[..., k][..., None]
        for k in range(nq - 1, -1, -1):
            x[..., k] = (x[..., k] - (A[..., k, k + 1:] * x[..., k + 1:]).sum(-1)) / A[..., k, k]
        psi[:, j, i] = x
    inv = [np.argsort(f[2]) for f in flips]
    return np.stack([psi[a][f[0], f[1]][..., inv[a]] for a, f in enumerate(flips)]).reshape(no, ny * nx, nq)


@pytest.mark.parametrize("p", [1, 2])
@pytest.mark.parametrize("nel,log_sd", [((8, 9), 1.0), ((40, 33), 1.0), ((61, 47), 0.0)])
def test_rows_are_accurate(nel, log_sd, p):
    """The 2-norm error against extended precision, next to that of the level kernel's LU."""
    print(f"rows accuracy {nel} p={p}", flush=True)
    rng = np.random.default_rng(7)
    ne = int(np.prod(nel))
    sig = P.lognormal_sigma(ne, log_sd, rng).reshape(1, -1)
    op = A.InverseAdvectionOperator(A.Mesh(nel), p, 4, sig)
    q = rng.uniform(0.5, 1.0, op.size) / ne
    ref = _extended_sweep(nel, p, op.quadrature()[0], sig[0], q.reshape(op.Nomega, ne, -1)).reshape(-1)
    err = {}
    for mode, lanes in ((0, 1), (3, 1)):
        op.set_tuning(mode, 64, lanes)
        psi = op.Mult(A.DeviceVector.from_host(q), A.DeviceVector(op.size)).to_host()
        err[mode] = float(np.sqrt(((psi - ref) ** 2).sum() / (ref ** 2).sum()))
    print(f"  LU {err[0]:.2e}  rows {err[3]:.2e}", flush=True)
    # Both accumulate the rounding errors of single cells.  At p = 1 the pair's unknowns are
    # three times as large as the trace they sum to, at p = 2 they are not larger than the
    # real one; the rest is room for chance, of which few cells of one direction have much.
    # A basis of condition 7 per axis (p = 2) gave 5 to 13 times the LU's error, constants
    # that err by 3e-16 in every element (p = 1) 5 to 10 times on the larger meshes.
    assert err[3] < (5.0 if p == 1 else 2.5) * err[0]


@pytest.mark.parametrize("nel,p", [((9, 70), 1), ((9, 70), 2), ((3, 4, 5), 2)])
def test_fp32_requests_that_run_fp64(nel, p):
    """2D rows and uniform 3D p = 2 cells serve FP32 requests in FP64, to the bit."""
    op = A.InverseAdvectionOperator(A.Mesh(nel), p, 4, np.ones((1, int(np.prod(nel)))))
    op.set_launch(3 if len(nel) == 2 else 0)
    q = A.DeviceVector.from_host(np.random.default_rng(1).uniform(0.1, 1.0, op.size))
    psi = [op.Mult(q, A.DeviceVector(op.size)).to_host()]
    op.set_precision(A.FP32_REFINED)
    psi.append(op.Mult(q, A.DeviceVector(op.size)).to_host())
    np.testing.assert_array_equal(*psi)


@pytest.mark.parametrize("p", [1, 2])
@pytest.mark.parametrize("nel,block", [((9, 5), 64), ((6, 150), 64)])
def test_rows_with_both_sources(nel, block, p):
    """A source per direction and an isotropic one together, as source iteration has them."""
    rng = np.random.default_rng(9)
    ne = int(np.prod(nel))
    sig = P.lognormal_sigma(2 * ne, 1.0, rng).reshape(2, ne)
    v = P.cartesian_vertices(nel, extents=(2.0, 1.0))
    op = A.InverseAdvectionOperator(A.Mesh(nel, vertices=v), p, 6, sig)
    op.set_tuning(3, block, 1)
    om, w = ls_fixture(6, 2)
    pr = oracle.Problem(2, nel, v, p, om, w, sig)
    q, iso = rng.uniform(0.1, 1.0, op.size), rng.uniform(0.1, 1.0, op.phi_size)
    ref = np.empty(op.size)
    pr.sweep(q + np.broadcast_to(iso.reshape(2, 1, -1), (2, op.Nomega, op.phi_size // 2)).reshape(-1), ref)
    psi, phi = A.DeviceVector.from_host(np.full(op.size, np.nan)), A.DeviceVector(op.phi_size)
    op.MultMoments(A.DeviceVector.from_host(q), psi, phi, A.DeviceVector.from_host(iso))
    # FP64 both, in other elimination orders; the moments sum positive terms
    assert rel_err(psi.to_host(), ref) < 1e-12
    assert rel_err(phi.to_host(), np.einsum("a,gai->gi", w, ref.reshape(2, op.Nomega, -1)).reshape(-1)) < 1e-12


# the traces of a strip's last row take 8 Q nx bytes of LDS next to 16 Q block of the lanes:
# 64 KB are 3968 elements at p = 1 and 2602 at p = 2 with 64 lanes
@pytest.mark.parametrize("nel,p,lump", [((3968, 65), 1, 0), ((3969, 65), 1, 0), ((2602, 65), 2, 0), ((2603, 65), 2, 0),
                                        ((12, 70), 1, 7), ((12, 70), 1, 1)])
def test_direction_sweeps_where_rows_stop(nel, p, lump):
    """Both sides of the LDS bound, and lumped matrices, which the rows do not take."""
    print(f"rows bound {nel} p={p} lump {lump}", flush=True)
    rng = np.random.default_rng(10)
    ne = int(np.prod(nel))
    sig = P.lognormal_sigma(ne, 1.0, rng).reshape(1, -1) * nel[0]
    # one direction per quadrant keeps the oracle short
    om = np.array([[0.7, 0.3], [-0.7, 0.3], [0.3, -0.7], [-0.3, -0.7]])
    w = np.full(4, 0.25)
    v = P.cartesian_vertices(nel)
    op = A.InverseAdvectionOperator(A.Mesh(nel, vertices=v), p, (om, w), sig, lump=lump)
    op.set_tuning(3, 64, 1)
    pr = oracle.Problem(2, nel, v, p, om, w, sig, lump=lump)
    q = rng.uniform(0.1, 1.0, op.size)
    ref = np.empty(op.size)
    pr.sweep(q, ref)
    psi = A.DeviceVector.from_host(np.full(op.size, np.nan))
    op.Mult(A.DeviceVector.from_host(q), psi)
    # relative to the largest value: FP64 both, in other elimination orders
    assert rel_err(psi.to_host(), ref) < 1e-12


@pytest.mark.parametrize("p", [1, 2])
def test_rows_along_the_axes(p):
    """Directions along an axis: one of t_x, t_y is zero."""
    nel, ne = (7, 66), 7 * 66
    sig = P.lognormal_sigma(ne, 1.0, np.random.default_rng(11)).reshape(1, -1)
    om = np.array([[1.0, 0.0], [-1.0, 0.0], [0.0, 1.0], [0.0, -1.0]])
    w = np.full(4, 0.25)
    op = A.InverseAdvectionOperator(A.Mesh(nel), p, (om, w), sig)
    op.set_tuning(3, 64, 1)
    pr = oracle.Problem(2, nel, P.cartesian_vertices(nel), p, om, w, sig)
    q = np.random.default_rng(12).uniform(0.1, 1.0, op.size)
    ref = np.empty(op.size)
    pr.sweep(q, ref)
    psi = op.Mult(A.DeviceVector.from_host(q), A.DeviceVector.from_host(np.full(op.size, np.nan)))
    # FP64 both, in other elimination orders
    assert rel_err(psi.to_host(), ref) < 1e-12
