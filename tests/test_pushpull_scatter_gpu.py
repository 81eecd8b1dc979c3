"""GPU parity of push / count on rotated and zoomed lattices of at least 2^20
samples, whose tiles outgrow the static LDS box and run in one or two larger
ones, against the FP64 oracle.

Tolerance: element-wise |gpu - oracle| <= 1e-4 * oracle(|v|) (+ 1e-36, below
float's normal range), as for the other routes.
"""
import numpy as np
import pytest
import torch

from oracle import pushpull as O

pytestmark = pytest.mark.gpu
DEV = "cuda"
BOUNDS = ["dct2", "dft", "zero", "dst1", "replicate", "dst2", "dct1", "dct2"]


def T(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def rotated(shape, deg, zoom):
    """Rotation about (1, 1, 1) by `deg` and a zoom about the centre."""
    k = np.ones(3) / np.sqrt(3)
    K = np.array([[0, -k[2], k[1]], [k[2], 0, -k[0]], [-k[1], k[0], 0]])
    t = np.deg2rad(deg)
    A = zoom * (np.eye(3) + np.sin(t) * K + (1 - np.cos(t)) * K @ K)
    c = (np.array(shape) - 1) / 2
    ijk = np.stack(np.meshgrid(*[np.arange(n, dtype=np.float64) for n in shape], indexing="ij"), -1)
    return ((ijk - c) @ A.T + c + np.array([0.3, -0.2, 0.1]))[None].astype(np.float32)


@pytest.mark.parametrize("order,deg,zoom", [(o, 15, 1.1) for o in (0, 1, 3, 5, 6)] + [(3, 30, 1.3)])
def test_rotated_push_count(order, deg, zoom):
    from nitorch_amd import grid as G
    rng = np.random.default_rng(2100 + order)
    shape = (102, 101, 103)
    bound, extrap = BOUNDS[order], (order + (deg > 15)) % 2
    g = rotated(shape, deg, zoom)
    g64 = g.astype(np.float64)
    y = rng.standard_normal((1, 2) + shape).astype(np.float32)
    y[0, 1, 50, 51, 52] = np.inf
    yt = T(np.moveaxis(y, 1, -1)).movedim(-1, 1)   # channel-last storage
    out = G.grid_push(yt, T(g), list(shape), [bound], [order], extrap).cpu().double().numpy()
    y64 = y.astype(np.float64)
    ref = O.grid_push(y64, g64, shape, bound, order, extrap, oob_f32=True)
    bar = O.grid_push(np.abs(y64), g64, shape, bound, order, extrap, oob_f32=True)
    fin = np.isfinite(ref)
    assert np.array_equal(np.isfinite(out), fin), ("non-finite", order, bound)
    if bound in ("dst1", "dst2"):   # signed folds cancel: no bar for an element, its largest for all
        bar = np.full(ref.shape, np.abs(bar[np.isfinite(bar)]).max())
    assert (np.abs(out[fin] - ref[fin]) <= 1e-4 * bar[fin] + 1e-36).all(), ("push", order, bound)
    out = G.grid_count(T(g), list(shape), [bound], [order], extrap).cpu().double().numpy()
    ref = O.grid_count(g64, shape, bound, order, extrap, oob_f32=True)
    bar = np.abs(ref).max() if bound in ("dst1", "dst2") else ref
    assert (np.abs(out - ref) <= 1e-4 * bar + 1e-36).all(), ("count", order, bound)
