"""Performance cases: what users of the sweep, the solvers, the radiation step and
the learned correction have them do, from the smallest calls to the largest.

``listed()`` names fixed cases, ``draw(rng)`` gives another one of the same
ranges, ``prepare`` makes the inputs and handles on the GPU, ``run`` is one pass
through the public entry points, ``work`` what the pass cannot do without,
``tolerance`` how far another correct implementation may be off, and ``exact``
the same outputs in plain 64-bit torch on the CPU.
"""
import ctypes
import math

import numpy as np
import torch
import torch.nn.functional as F

import allium_amd as A
from allium_amd import _lib, cnn, trt
from allium_amd import problems as P


def listed():
    return [
        # the 2D one-group deck on 32 x 32 quads: one inversion is a few hundred
        # small dependent steps, so latency and launches are what counts
        _sweep("sweep_2d_p1_32", 32, 32, 1, 1, 8),
        # a quadratic 2D run on a mesh that no tile divides
        _sweep("sweep_2d_p2_150x97", 150, 97, 1, 2, 12),
        # the headline sweep: 64^3 hexes, 80 directions, 1.7e8 unknowns
        _sweep("sweep_3d_p1_64", 64, 64, 64, 1, 8),
        # a distorted mesh: every element and face has matrices of its own
        _sweep("sweep_3d_p1_jittered", 26, 23, 29, 1, 8, jitter=0.05),
        # uneven quadratic instances swept together, distorted meshes, S12
        {"name": "batch_3d_p2_jittered", "kind": "batch", "n1": 16, "n2": 18, "n3": 21, "sn": 12},
        # the inner step of a multigroup solver: isotropic source in, scalar flux out
        _sweep("moments_3d_4_groups", 30, 25, 37, 1, 6, groups=4, moments=True),
        # the 2D deck solved by source iteration to 1e-8: many tiny sweeps
        _solve("si_2d_p1_32", "si", 32, 32, 1, 0.9, 0.0, 1.0),
        # highly scattering heterogeneous 3D medium, Krylov outer solver
        _solve("gmres_3d_p1_32", "gmres", 32, 32, 32, 0.9999, 1.5, 1.0),
        # thick scattering medium, source iteration with diffusion acceleration
        _solve("dsa_3d_p1_thick", "dsa", 28, 24, 33, 0.999, 1.0, 10.0),
        # one backward-Euler step of multigroup thermal radiation, 16 groups
        {"name": "trt_3d_16_groups", "kind": "trt", "nx": 20, "ny": 16, "nz": 18, "sn": 6, "groups": 16},
        # the correction network on a 64^3 grid, as a solve on that mesh applies it
        {"name": "cnn_forward_64", "kind": "forward", "batch": 1, "nz": 64, "ny": 64, "nx": 64},
        # one training step on a batch of 32^3 grids, forward, backward and Adam
        {"name": "cnn_train_8x32", "kind": "train", "batch": 8, "nz": 32, "ny": 32, "nx": 32},
    ]


def _sweep(name, nx, ny, nz, p, sn, groups=1, jitter=0.0, fp32=False, moments=False):
    c = {"kind": "sweep", "nx": nx, "ny": ny, "nz": nz, "p": p, "sn": sn, "groups": groups, "jitter": jitter,
         "fp32": fp32, "moments": moments}
    return dict(c, name=name) if name else c


def _solve(name, solver, nx, ny, nz, c, log_sd, scale):
    d = {"kind": "solve", "solver": solver, "nx": nx, "ny": ny, "nz": nz, "p": 1, "sn": 8, "groups": 1,
         "jitter": 0.0, "c": c, "log_sd": log_sd, "scale": scale}
    return dict(d, name=name) if name else d


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["sweep"] * 5 + ["batch", "moments", "solve", "solve", "trt", "forward", "train"])
    if kind in ("sweep", "moments"):
        jitter = 0.05 if kind == "sweep" and rng.random() < 0.3 else 0.0
        fp32 = rng.random() < 0.15
        groups = rng.choice([1, 1, 1, 2, 3, 8])
        if rng.random() < 0.4:
            return _sweep(None, _log(rng, 8, 300), _log(rng, 8, 300), 1, rng.choice([0, 1, 1, 2]),
                          rng.choice([4, 8, 12]), groups, jitter, fp32, kind == "moments")
        m = 26 if jitter or groups > 1 else 56
        return _sweep(None, _log(rng, 4, m), _log(rng, 4, m), _log(rng, 4, m), rng.choice([0, 1, 1, 1]),
                      rng.choice([4, 6, 8]), groups, jitter, fp32, kind == "moments")
    if kind == "batch":
        return {"kind": "batch", "n1": rng.randint(8, 20), "n2": rng.randint(8, 20), "n3": rng.randint(8, 20),
                "sn": rng.choice([8, 12])}
    if kind == "solve":
        solver = rng.choice(["si", "gmres", "fgmres", "dsa"])
        c = {"si": rng.uniform(0.5, 0.95), "dsa": rng.uniform(0.99, 0.9999)}.get(solver, rng.uniform(0.9, 0.9999))
        scale = rng.uniform(1.0, 20.0) if solver == "dsa" else 1.0
        if rng.random() < 0.5:
            d = _solve(None, solver, _log(rng, 8, 100), _log(rng, 8, 100), 1, c, rng.uniform(0, 1.5), scale)
        else:
            d = _solve(None, solver, _log(rng, 5, 30), _log(rng, 5, 30), _log(rng, 5, 30), c, rng.uniform(0, 1.5),
                       scale)
        return dict(d, sn=rng.choice([4, 8]))
    if kind == "trt":
        return {"kind": "trt", "nx": rng.randint(5, 18), "ny": rng.randint(5, 18), "nz": rng.randint(5, 18),
                "sn": rng.choice([4, 6]), "groups": rng.choice([4, 8, 16])}
    if kind == "forward":
        return {"kind": "forward", "batch": 1, "nz": _log(rng, 8, 64), "ny": _log(rng, 8, 64), "nx": _log(rng, 8, 64)}
    return {"kind": "train", "batch": rng.randint(1, 8), "nz": rng.randint(9, 32), "ny": rng.randint(9, 32),
            "nx": rng.randint(9, 32)}


# ---------------------------------------------------------------- inputs, from the seed alone

def _nel(case):
    return (case["nx"], case["ny"]) if case["nz"] == 1 else (case["nx"], case["ny"], case["nz"])


def _medium(case, seed):
    """(elements per axis, vertices or None, sigma_t (G, Ne), sigma_s (Ne,))"""
    rng = np.random.default_rng(seed)
    nel = _nel(case)
    ne = int(np.prod(nel))
    vert = P.jittered_vertices(nel, case["jitter"], rng) if case["jitter"] else None
    sig = np.stack([P.lognormal_sigma(ne, case.get("log_sd", 1.0), rng) for _ in range(case["groups"])])
    sig *= case.get("scale", 1.0) * rng.uniform(0.95, 1.05)
    return nel, vert, sig, case.get("c", 0.9) * sig[0]


def _phi_source(nel, p, groups, seed, device):
    """An isotropic source like an integrated fission or emission density: lognormal
    per element, a little variation between its nodes, times the nodes' share
    of the element's volume.  (G, Ne, n)"""
    g = torch.Generator(device="cpu").manual_seed(int(seed))
    ne, dim = int(np.prod(nel)), len(nel)
    w1 = {0: [1.0], 1: [0.5, 0.5], 2: [1 / 6, 2 / 3, 1 / 6]}[p]
    w = torch.tensor(w1, dtype=torch.float64)
    for _ in range(dim - 1):
        w = torch.outer(w, torch.tensor(w1, dtype=torch.float64)).reshape(-1)
    q = torch.exp(0.5 * torch.randn(groups, ne, 1, generator=g, dtype=torch.float64))
    q = q * (1.0 + 0.1 * torch.rand(groups, ne, w.numel(), generator=g, dtype=torch.float64)) * w / ne
    return q.to(device)


def _psi_source(iso, weights):
    """The source of every direction: the isotropic one, tilted by the direction
    so that no two directions are alike.  (G, Nomega, Ne, n)"""
    t = torch.linspace(0.7, 1.3, len(weights), dtype=torch.float64, device=iso.device)
    return t[None, :, None, None] * iso[:, None]


def _grids(case, seed):
    g = np.random.default_rng(seed)
    shape = (case["batch"], case["nz"], case["ny"], case["nx"])
    x = g.standard_normal(shape + (3,), dtype=np.float32)
    x[..., 2] = g.uniform(0.9, 1.0, shape)
    return x, g.standard_normal(shape, dtype=np.float32) * np.float32(0.5)


def _net_params(seed):
    """He-normal weights, small biases: (packed float32)"""
    g, out = np.random.default_rng(seed + 77), []
    for ci, co in zip(_CH[:-1], _CH[1:]):
        out += [g.standard_normal(27 * co * ci) * math.sqrt(2.0 / (27 * ci)), g.standard_normal(co) * 0.01]
    return np.concatenate(out).astype(np.float32)


_CH = [3, 32, 32, 32, 32, 1]


class _Vector(A.DeviceVector):
    """A torch tensor's memory as the library's device vector."""

    def __init__(self, t):
        self.t, self.n, self.ptr = t, t.numel(), ctypes.c_void_p(t.data_ptr())

    def free(self):
        self.ptr = None


_tuned = {}


def _tune(op, key):
    """Autotune the first handle of a shape; later ones take its launch
    settings over, as a program with many handles does."""
    if key not in _tuned:
        op.set_launch(-1)
        t = op.tuning()
        _tuned[key] = (t, op.box_tiling() if t["mode"] >= 4 else None)
        return
    t, box = _tuned[key]
    if box:
        op.set_box_tiling(box["bx"], box["by"], box["bz"], box["dirs_per_group"], box["threads"], box["prefetch"])
    op.set_tuning(t["mode"], t["block"], t["lanes"])


def _operator(case, seed):
    nel, vert, sig, sigma_s = _medium(case, seed)
    op = A.InverseAdvectionOperator(A.Mesh(nel, vertices=vert), case["p"], case["sn"], sig,
                                    precision=A.FP32_REFINED if case.get("fp32") else A.FP64)
    _tune(op, str(sorted((k, v) for k, v in case.items() if k != "name")))
    return op, sigma_s


def prepare(case, seed):
    if case["kind"] == "sweep":
        op, _ = _operator(case, seed)
        iso = _phi_source(_nel(case), case["p"], case["groups"], seed, "cuda")
        psi = torch.empty(op.size, dtype=torch.float64, device="cuda")
        s = {"op": op, "psi": _Vector(psi)}
        if case["moments"]:
            s["iso"] = _Vector(iso.contiguous())
            s["phi"] = _Vector(torch.empty(op.phi_size, dtype=torch.float64, device="cuda"))
        else:
            s["q"] = _Vector(_psi_source(iso, op.quadrature()[1]).contiguous())
        return s
    if case["kind"] == "batch":
        ops, isos, psis = [], [], []
        for i, n in enumerate((case["n1"], case["n2"], case["n3"])):
            c = _batch_member(case, n)
            nel, vert, sig, _ = _medium(c, seed + 1000 * i)
            ops.append(A.InverseAdvectionOperator(A.Mesh(nel, vertices=vert), 2, case["sn"], sig))
            isos.append(_Vector(_phi_source(nel, 2, 1, seed + 1000 * i, "cuda").contiguous()))
            psis.append(_Vector(torch.empty(ops[-1].size, dtype=torch.float64, device="cuda")))
        return {"batch": A.SweepBatch(ops), "isos": isos, "psis": psis}
    if case["kind"] == "solve":
        op, sigma_s = _operator(case, seed)
        iso = _phi_source(_nel(case), 1, 1, seed, "cuda")
        s = {"op": op, "sigma_s": sigma_s, "solver": case["solver"],
             "q": _Vector(_psi_source(iso, op.quadrature()[1]).contiguous())}
        if case["solver"] == "dsa":
            s["dsa"] = A.DSA(op, sigma_s)
        return s
    if case["kind"] == "trt":
        rng = np.random.default_rng(seed)
        t = trt.TRT((case["nx"], case["ny"], case["nz"]), sn=case["sn"], groups=case["groups"],
                    opacity_coef=rng.uniform(8.0, 12.0), T0=rng.uniform(0.01, 0.02), T_inflow=rng.uniform(0.9, 1.1))
        t.set_launch(-1)
        return {"trt": t}
    net = cnn.FluxCorrector(0, dilation=cnn.DILATION)
    net.set_params(_net_params(seed))
    x, target = _grids(case, seed)
    s = {"net": net, "shape": x.shape[:4], "x": cnn.DeviceArray32(x)}
    if case["kind"] == "train":
        s["target"] = cnn.DeviceArray32(target)
    else:
        s["out"] = torch.empty(x.shape[:4], dtype=torch.float32, device="cuda")
    return s


def _batch_member(case, n):
    return {"nx": n, "ny": n, "nz": n, "p": 2, "sn": case["sn"], "groups": 1, "jitter": 0.05}


def run(s):
    if "batch" in s:
        s["batch"].Mult(None, s["psis"], s["isos"])
        return [v.t for v in s["psis"]]
    if "trt" in s:
        s["trt"].step()
        return {"T": s["trt"].temperature(), "phi": s["trt"].scalar_flux()}
    if "net" in s:
        if "target" in s:
            loss = s["net"].train_step(s["x"], s["target"], s["shape"], 1e-3)
            return {"loss": loss, "params": s["net"].params()}
        _lib.check(_lib.load().allium_cnn_forward_device(s["net"].handle, *s["shape"], s["x"].ptr,
                                                         ctypes.c_void_p(s["out"].data_ptr()), None))
        return s["out"]
    if "iso" in s:
        s["op"].MultMoments(None, s["psi"], s["phi"], s["iso"])
        return {"psi": s["psi"].t, "phi": s["phi"].t}
    if "solver" not in s:
        s["op"].Mult(s["q"], s["psi"])
        return s["psi"].t
    if s["solver"] in ("si", "dsa"):
        return A.source_iteration(s["op"], s["sigma_s"], s["q"], abstol=1e-8, maxit=2000, want_psi=False,
                                  accel=s.get("dsa"))[0]
    return A.krylov_solve(s["op"], s["sigma_s"], s["q"], solver=s["solver"], abstol=1e-8, maxit=500,
                          want_psi=False)[0]


# ---------------------------------------------------------------- what a pass cannot do without

def _sweep_work(ne, dim, p, nomega, groups, jitter, psi_in=True):
    """Reading the source, writing psi, and each element's data once; per cell the
    upwind face terms and the local solve (dense elimination where every element
    has its own matrix, the tensor-product solve on a uniform mesh)."""
    n, nf = (p + 1) ** dim, (p + 1) ** (dim - 1)
    cells = ne * nomega * groups
    b = 8.0 * cells * n * (2 if psi_in else 1) + 8.0 * ne * groups
    if not jitter:
        return b, cells * n * (4.0 * dim + 2.0 * dim * (p + 1))
    b += 8.0 * ne * ((dim + 1) * n * n + dim * nf * nf + 3 * dim)
    return b, cells * (2.0 * n ** 3 / 3 + 2.0 * (dim + 1) * n * n + 2.0 * n * n + 4.0 * dim * nf * nf)


def _nomega(sn, dim):
    return sn * (sn + 2) // (1 if dim == 3 else 2)


def work(case):
    if case["kind"] == "batch":
        ws = [_sweep_work(n ** 3, 3, 2, _nomega(case["sn"], 3), 1, True, False)
              for n in (case["n1"], case["n2"], case["n3"])]
        return {"bytes": sum(w[0] for w in ws), "flops": sum(w[1] for w in ws)}
    if case["kind"] in ("forward", "train"):
        vox = case["batch"] * case["nz"] * case["ny"] * case["nx"]
        macs = vox * 27.0 * sum(a * b for a, b in zip(_CH[:-1], _CH[1:]))
        if case["kind"] == "forward":
            return {"bytes": 16.0 * vox, "flops": 2.0 * macs}
        return {"bytes": 16.0 * vox + 2 * 2 * 128.0 * vox, "flops": 6.0 * macs}
    if case["kind"] == "trt":
        ne = case["nx"] * case["ny"] * case["nz"]
        b, f = _sweep_work(ne, 3, 1, _nomega(case["sn"], 3), case["groups"], False, False)
        # the first and the last sweep read psi-sized sources, about three iterations between them
        return {"bytes": 8.0 * b, "flops": 5.0 * f}
    nel = _nel(case)
    ne, dim = int(np.prod(nel)), len(nel)
    nom = _nomega(case["sn"], dim)
    b, f = _sweep_work(ne, dim, case["p"], nom, case["groups"], case["jitter"] > 0,
                       case["kind"] == "sweep" and not case["moments"])
    if case["kind"] == "sweep":
        return {"bytes": b, "flops": f}
    # one sweep with the source and as many without it as the method takes on such media
    its = {"si": 8.0 / -math.log10(0.6 * case["c"]), "dsa": 12.0, "gmres": 15.0, "fgmres": 15.0}[case["solver"]]
    return {"bytes": b * its, "flops": f * its}


def tolerance(case):
    if case["kind"] == "forward":
        return {"rel": 2e-2, "max": 0.5}     # bfloat16 activations
    if case["kind"] == "train":
        # the first Adam step moves a weight by the rate whichever way its gradient points
        return {"rel": 5e-3, "max": 0.2}
    if case["kind"] == "trt":
        return {"rel": 1e-8, "max": 1e-5}    # stops its iteration at 1e-8 of the first change
    if case["kind"] == "solve":
        # stop at a change or residual of 1e-8; the diffusion solve inside stops at 1e-6
        return {"rel": 1e-9, "max": 1e-7} if case["solver"] == "si" else {"rel": 1e-7, "max": 1e-5}
    if case.get("fp32"):
        return {"rel": 1e-5, "max": 1e-3}    # 32-bit cell solves, about 2e-6 measured
    return {"rel": 1e-13, "max": 1e-11}      # 64-bit throughout, about 1e-14 measured


# ---------------------------------------------------------------- the same in plain 64-bit torch

def exact(case, seed):
    if case["kind"] in ("forward", "train"):
        return _exact_net(case, seed)
    if case["kind"] == "trt":
        return None     # tens of millions of cell solves a step
    if case["kind"] == "batch":
        cases = [_batch_member(case, n) for n in (case["n1"], case["n2"], case["n3"])]
        if sum(_cost(c) for c in cases) > 12:
            return None
        out = []
        for i, c in enumerate(cases):
            nel, vert, sig, _ = _medium(c, seed + 1000 * i)
            iso = _phi_source(nel, 2, 1, seed + 1000 * i, "cpu")
            out.append(_Transport(c, nel, vert, sig).sweep(iso[:, None].expand(-1, _nomega(case["sn"], 3), -1, -1))
                       .reshape(-1))
        return out
    if _cost(case) * (25 if case["kind"] == "solve" else 1) > 15:
        return None
    nel, vert, sig, sigma_s = _medium(case, seed)
    tr = _Transport(case, nel, vert, sig)
    iso = _phi_source(nel, case["p"], case["groups"], seed, "cpu")
    if case["kind"] == "sweep":
        if case["moments"]:
            psi = tr.sweep(iso[:, None].expand(-1, len(tr.w), -1, -1))
            return {"psi": psi.reshape(-1), "phi": torch.einsum("a,gaei->gei", tr.w, psi).reshape(-1)}
        return tr.sweep(_psi_source(iso, tr.w)).reshape(-1)
    return tr.solve(torch.from_numpy(sigma_s), _psi_source(iso, tr.w)).reshape(-1).numpy()


def _cost(case):
    """Seconds that a plain sweep takes, roughly."""
    nel = _nel(case)
    dim = len(nel)
    n = (case["p"] + 1) ** dim
    return float(np.prod(nel)) * _nomega(case["sn"], dim) * case["groups"] * (2e-6 + 1.3e-9 * n ** 3)


def _gauss(m):
    x, w = np.polynomial.legendre.leggauss(m)
    return (x + 1) / 2, w / 2


def _tensor_points(dim, m):
    """Gauss points (q, 3) and weights of the unit cube, first axis fastest."""
    x, w = _gauss(m)
    g = np.meshgrid(*[x] * dim, indexing="ij")
    pts = np.stack([a.transpose(*reversed(range(dim))).reshape(-1) for a in g], 1) if dim else np.zeros((1, 0))
    wt = np.ones(1)
    for _ in range(dim):
        wt = np.outer(w, wt).reshape(-1)
    return pts, wt


def _basis(nodes, pts):
    """Tensor Lagrange basis at pts (q, dim): values (q, n), gradients (q, n, dim)."""
    k, dim = len(nodes), pts.shape[1]
    v = np.ones((dim, len(pts), k))
    d = np.zeros((dim, len(pts), k))
    for a in range(dim):
        for i in range(k):
            others = [m for m in range(k) if m != i]
            v[a, :, i] = np.prod([(pts[:, a] - nodes[m]) / (nodes[i] - nodes[m]) for m in others], axis=0)
            for r in others:
                rest = [(pts[:, a] - nodes[m]) / (nodes[i] - nodes[m]) for m in others if m != r]
                d[a, :, i] += np.prod(rest, axis=0) / (nodes[i] - nodes[r])
    val, grad = np.ones((len(pts), 1)), np.ones((len(pts), 1, dim))
    for a in range(dim):
        val = (v[a][:, :, None] * val[:, None, :]).reshape(len(pts), -1)
        f = np.stack([d[a] if a == b else v[a] for b in range(dim)], -1)
        grad = (f[:, :, None, :] * grad[:, None, :, :]).reshape(len(pts), -1, dim)
    return val, grad


class _Transport:
    """DG upwind transport on a structured mesh by dense local solves: cells in
    dependency order, all that are ready at a time."""

    def __init__(self, case, nel, vert, sig):
        self.nel, self.p, self.dim = nel, case["p"], len(nel)
        dim, p, ne = self.dim, self.p, int(np.prod(nel))
        self.om, w = A.level_symmetric(case["sn"], dim)
        self.w, self.sig = torch.from_numpy(w), torch.from_numpy(sig)
        self.nodes = {0: [0.5], 1: [0.0, 1.0], 2: [0.0, 0.5, 1.0]}[p]
        self.n, self.nf = (p + 1) ** dim, (p + 1) ** (dim - 1)
        v = (P.cartesian_vertices(nel) if vert is None else vert).reshape(*reversed([k + 1 for k in nel]), dim)
        corners = []
        for c in range(1 << dim):
            sl = tuple(slice((c >> d) & 1, ((c >> d) & 1) + nel[d]) for d in reversed(range(dim)))
            corners.append(v[sl].reshape(-1, dim))
        self.corners = np.stack(corners, 1)                       # (Ne, 2^dim, dim)
        self.vert_basis = lambda pts: _basis([0.0, 1.0], pts)
        self._element_matrices()
        self._faces()
        self.ne = ne
        self._order()

    def _jac(self, pts):
        g = self.vert_basis(pts)[1]                               # (q, 2^dim, dim)
        return np.einsum("ecm,qcd->eqmd", self.corners, g)        # dX_m / dxi_d

    def _element_matrices(self):
        dim, p = self.dim, self.p
        pts, wt = _tensor_points(dim, (2 * p) // 2 + 1)
        phi = _basis(self.nodes, pts)[0]
        self.M = torch.from_numpy(np.einsum("eq,qi,qj->eij", np.linalg.det(self._jac(pts)) * wt, phi, phi,
                                            optimize=True))
        pts, wt = _tensor_points(dim, (dim + 2 * p - 1) // 2 + 1)
        phi, dphi = _basis(self.nodes, pts)
        J = self._jac(pts)
        adj = np.linalg.inv(J) * np.linalg.det(J)[..., None, None]
        self.Gd = torch.from_numpy(-np.einsum("q,qir,eqrd,qj->edij", wt, dphi, adj, phi, optimize=True))

    def _faces(self):
        """Per element and side: outward unit normal at the side's centre, face mass
        in face-local numbering, neighbour, nodes."""
        dim, p, nel = self.dim, self.p, self.nel
        ne = int(np.prod(nel))
        idx = np.arange(ne).reshape(*reversed(nel))
        fp, fw = _tensor_points(dim - 1, (2 * p) // 2 + 1)
        self.nor = np.zeros((ne, 2 * dim, dim))
        self.Fm, self.nb, self.side = [], np.full((ne, 2 * dim), -1), []
        local = np.stack(np.unravel_index(np.arange(self.n), [p + 1] * dim)[::-1], 1)
        for s in range(2 * dim):
            ax, hi = s >> 1, s & 1
            at = np.insert(fp, ax, float(hi), axis=1)
            area, _ = self._surface(at, ax, hi)
            phi = _basis(self.nodes, at)[0]
            nodes = np.nonzero(local[:, ax] == (p if hi else 0))[0]
            self.side.append(nodes)
            self.Fm.append(torch.from_numpy(np.einsum("eq,qk,ql->ekl", area * fw, phi[:, nodes], phi[:, nodes],
                                                      optimize=True)))
            mid = np.insert(np.full((1, dim - 1), 0.5), ax, float(hi), axis=1)
            self.nor[:, s] = self._surface(mid, ax, hi)[1][:, 0]
            lo_sl, hi_sl = [slice(None)] * dim, [slice(None)] * dim
            lo_sl[dim - 1 - ax], hi_sl[dim - 1 - ax] = slice(0, -1), slice(1, None)
            a, b = idx[tuple(lo_sl)].reshape(-1), idx[tuple(hi_sl)].reshape(-1)
            if hi:
                self.nb[a, s] = b
            else:
                self.nb[b, s] = a
        for s in range(1, 2 * dim, 2):      # one normal and mass per face: the low element's
            e = np.nonzero(self.nb[:, s] >= 0)[0]
            self.nor[self.nb[e, s], s - 1] = -self.nor[e, s]
            self.Fm[s - 1][self.nb[e, s]] = self.Fm[s][e]
        self.dot = np.einsum("ad,esd->aes", self.om, self.nor)

    def _surface(self, pts, ax, hi):
        """Area element and outward unit normal of a side at pts."""
        J = self._jac(pts)
        adj = np.linalg.inv(J) * np.linalg.det(J)[..., None, None]
        v = adj[:, :, ax, :] * (1.0 if hi else -1.0)
        area = np.linalg.norm(v, axis=-1)
        return area, v / area[..., None]

    def _order(self):
        """Levels of (direction, element) pairs: each after all that it reads."""
        na, ne, ns = len(self.om), self.ne, 2 * self.dim
        need = (self.dot < 0) & (self.nb >= 0)[None]
        wait = need.sum(-1)
        self.levels = []
        a, e = np.nonzero(wait == 0)
        left = na * ne
        while len(a):
            self.levels.append((a, e))
            left -= len(a)
            nxt = []
            for s in range(ns):
                o = self.nb[e, s]
                k = o >= 0
                k[k] = need[a[k], o[k], s ^ 1]
                wait[a[k], o[k]] -= 1
                nxt.append((a[k], o[k]))
            key = np.unique(np.concatenate([x * ne + y for x, y in nxt]))
            key = key[wait[key // ne, key % ne] == 0]
            a, e = key // ne, key % ne
        if left:
            raise RuntimeError("cyclic sweep graph")

    def _matrix(self, g, a, e):
        K = self.sig[g, e, None, None] * self.M[e]
        om = torch.from_numpy(self.om[a])
        for d in range(self.dim):
            K = K + om[:, d, None, None] * self.Gd[e, d]
        for s in range(2 * self.dim):
            w = torch.from_numpy(np.maximum(self.dot[a, e, s], 0.0))
            n = torch.from_numpy(self.side[s])
            K[:, n[:, None], n[None, :]] += w[:, None, None] * self.Fm[s][e]
        return K

    def sweep(self, q, keep=None):
        """psi = L^{-1} q, q (G, Nomega, Ne, n); `keep`: a dict that takes the inverses."""
        psi = torch.zeros(q.shape, dtype=torch.float64)
        for g in range(q.shape[0]):
            for L, (a, e) in enumerate(self.levels):
                for i in range(0, len(a), 100000):
                    self._cells(psi, q, g, a[i:i + 100000], e[i:i + 100000], keep, (g, L, i))
        return psi

    def _cells(self, psi, q, g, a, e, keep, key):
        at, et = torch.from_numpy(a), torch.from_numpy(e)
        b = q[g, at, et].clone()
        for s in range(2 * self.dim):
            dot = self.dot[a, e, s]
            o = self.nb[e, s]
            inner = (dot < 0) & (o >= 0)
            mine, other = torch.from_numpy(self.side[s]), torch.from_numpy(self.side[s ^ 1])
            u = torch.zeros(len(a), self.nf, dtype=torch.float64)
            k = torch.from_numpy(np.nonzero(inner)[0])
            u[k] = psi[g, at[k], torch.from_numpy(o)[k]][:, other]
            f = torch.matmul(self.Fm[s][et], u[:, :, None])[:, :, 0]
            b[:, mine] += torch.from_numpy(np.maximum(-dot, 0.0))[:, None] * f
        if keep is None:
            psi[g, at, et] = torch.linalg.solve(self._matrix(g, a, e), b)
            return
        if key not in keep:
            keep[key] = torch.linalg.inv(self._matrix(g, a, e))
        psi[g, at, et] = torch.matmul(keep[key], b[:, :, None])[:, :, 0]

    def solve(self, sigma_s, q):
        """The scalar flux of (L - D^T Ms D) psi = q, by restarted GMRES on it."""
        pts, wt = _tensor_points(self.dim, (2 * self.p + self.dim - 1) // 2 + 1)
        phi = _basis(self.nodes, pts)[0]
        Ms = torch.from_numpy(np.einsum("eq,qi,qj->eij", np.linalg.det(self._jac(pts)) * wt, phi, phi, optimize=True))
        Ms = sigma_s[:, None, None] * Ms / self.w.sum()
        keep = {}

        def flux(src):
            return torch.einsum("a,gaei->gei", self.w, self.sweep(src, keep)).reshape(-1)

        def op(x):
            y = torch.matmul(Ms, x.reshape(self.ne, self.n, 1)).reshape(1, 1, self.ne, self.n)
            return x - flux(y.expand(-1, len(self.w), -1, -1))

        b = flux(q)
        x, r = torch.zeros_like(b), b
        for _ in range(20):
            beta = float(r.norm())
            if beta < 1e-14 * float(b.norm()):
                break
            V, H = [r / beta], np.zeros((21, 20))
            for j in range(20):
                w = op(V[j])
                for _ in range(2):
                    for i in range(j + 1):
                        h = float(V[i] @ w)
                        H[i, j] += h
                        w = w - h * V[i]
                H[j + 1, j] = float(w.norm())
                if H[j + 1, j] < 1e-15 * beta:
                    break
                V.append(w / H[j + 1, j])
            m = j + 1
            y = np.linalg.lstsq(H[:m + 1, :m], np.eye(m + 1)[0] * beta, rcond=None)[0]
            x = x + sum(float(y[i]) * V[i] for i in range(m))
            r = b - op(x)
        return x


def _exact_net(case, seed):
    x, target = _grids(case, seed)
    p = torch.from_numpy(_net_params(seed)).double().requires_grad_(case["kind"] == "train")
    a = torch.from_numpy(x).double().permute(0, 4, 1, 2, 3)
    i = 0
    for l, (ci, co) in enumerate(zip(_CH[:-1], _CH[1:])):
        W = p[i:i + 27 * co * ci].reshape(3, 3, 3, co, ci).permute(3, 4, 0, 1, 2)
        i += 27 * co * ci
        a = F.conv3d(a, W, p[i:i + co], padding=cnn.DILATION[l], dilation=cnn.DILATION[l])
        i += co
        a = F.relu(a) if l < 4 else a
    out = a[:, 0]
    if case["kind"] == "forward":
        return out
    loss = ((out - torch.from_numpy(target).double()) ** 2).mean()
    loss.backward()
    g = p.grad
    return {"loss": loss.item(), "params": (p.detach() - 1e-3 * g / (g.abs() + 1e-8)).numpy()}
