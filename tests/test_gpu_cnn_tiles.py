"""Tilings and row chains of the network kernels at their edges.

The convolutions take 8^3 or 4^3 voxel tiles of a dilation sub-grid, the weight
gradients chains of rows one dilation apart in chunks of 32 voxels: shapes on
both sides of each tile, chunk and chain boundary, against the FP64 oracle with
the same bfloat16 rounding points.  What differs is the FP32 summation order
(forward: 864 products, 2^-24 sqrt(864) = 2e-6) and the bfloat16 roundings that
it flips, 2^-8 relative in each of five layers: 5e-3 forward, 2e-2 for the
gradients (L2), as a flipped rounding in every layer of both passes would give.
"""
import numpy as np
import pytest

from allium_amd import cnn
from oracle import cnn_oracle as C

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float(np.linalg.norm(np.ravel(a) - np.ravel(b)) / max(np.linalg.norm(np.ravel(b)), 1e-300))


@pytest.mark.parametrize("shape,dil", [
    ((1, 17, 5, 33), (8, 4, 3, 8, 5)),    # small tiles, several along x and z
    ((1, 4, 9, 40), (1, 2, 8, 1, 8)),     # both kinds; chains of one and two rows
    ((2, 1, 1, 1), (1, 8, 2, 1, 4)),      # one voxel
    ((1, 2, 3, 65), (7, 1, 1, 6, 2)),     # three chunks of a row, fewer rows than residues
])
def test_tiles_and_chains_match_oracle(shape, dil):
    print(f"cnn tiles {shape} {dil}", flush=True)
    rng = np.random.default_rng(21)
    params = [(W, rng.normal(0, 0.05, b.shape)) for W, b in C.init_params(22)]
    flat32 = C.pack(params).astype(np.float32)
    p32 = C.unpack(flat32.astype(np.float64))
    net = cnn.FluxCorrector(0, dilation=dil)
    net.set_params(flat32)
    x = rng.normal(size=shape + (3,)).astype(np.float32)
    t = rng.normal(size=shape).astype(np.float32)
    ref, _ = C.forward(p32, x.astype(np.float64), bf16=True, dil=list(dil))
    assert _rel(net.forward(x), ref) < 5e-3
    _, grads = C.loss_and_grad(p32, x.astype(np.float64), t.astype(np.float64), bf16=True, dil=list(dil))
    _, g = net.gradient(x, t)
    for l, ((gW, gb), (rW, rb)) in enumerate(zip(C.unpack(g.astype(np.float64)), grads)):
        assert _rel(gW, rW) < 2e-2 and _rel(gb, rb) < 2e-2, l
