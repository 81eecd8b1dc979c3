"""GPU checks of pulls at the limits of what their entry points take:
extrapolated coordinates beyond the integer range or infinite, whose first
taps saturate, and source views with negative strides (C ABI).

Tolerance against the FP64 oracle: 1e-5 norm-relative, as the other gathers
(float sums of at most (order + 1)^3 terms)."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import pushpull as O

pytestmark = pytest.mark.gpu


def T(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def close(a, b):
    a = a.detach().cpu().double().numpy()
    return np.abs(a - b).max() <= 1e-5 * np.abs(b).max()


@pytest.mark.parametrize("value", [3e9, 1e10, -1e10, np.inf, -np.inf])
@pytest.mark.parametrize("axes", [(0,), (1,), (2,), (0, 1, 2)])
@pytest.mark.parametrize("order", [1, 2, 3])
def test_gather_beyond_the_integer_range(order, axes, value):
    """Tiles of 4 x 8 x 16 samples: the first is ordinary, every sample of the
    second lies at `value` along `axes`.  Under `zero` its finite coordinates
    read as zero (weights stay finite up to order 3)."""
    from nitorch_amd import grid as G
    rng = np.random.default_rng(order)
    shape, source = (4, 8, 32), (9, 10, 40)
    g = np.stack(np.meshgrid(*[np.arange(n, dtype=np.float64) + 2 for n in shape], indexing="ij"), -1)[None]
    g = (g + rng.uniform(-0.6, 0.6, g.shape)).astype(np.float32)
    for d in axes:
        g[:, :, :, 16:, d] = value
    x = rng.standard_normal((1, 4) + source).astype(np.float32)
    u = rng.standard_normal((1, 4) + shape).astype(np.float32)
    first = (Ellipsis, slice(0, 16))
    g64, x64, u64 = (t.astype(np.float64) for t in (g[:, :, :, :16], x, u[first]))
    for bound in ("zero", "dct1", "dct2", "dst1", "dst2", "dft", "replicate"):
        pull = G.grid_pull(T(x), T(g), [bound], [order], 1)
        grad = G.grid_grad(T(x), T(g), [bound], [order], 1)
        ggrad, = G.grid_pull_backward(T(u), T(x), T(g).requires_grad_(), [bound], [order], 1)
        assert close(pull[first], O.grid_pull(x64, g64, bound, order, 1, oob_f32=True)), bound
        assert close(grad[:, :, :, :, :16], O.grid_grad(x64, g64, bound, order, 1, oob_f32=True)), bound
        ref = O.grid_pull_backward(u64, x64, g64, bound, order, 1, oob_f32=True)[1]
        assert close(ggrad[:, :, :, :16], ref), bound
        if bound == "zero" and np.isfinite(value):
            assert not pull[..., 16:].any() and not grad[:, :, :, :, 16:].any() and not ggrad[:, :, :, 16:].any()


@pytest.mark.parametrize("order", [1, 2, 3])
def test_bins_beyond_the_integer_range(order):
    """Calls large enough for the binned second pass, with samples beyond the
    integer range and infinite in every tile: under `zero` they add and read
    nothing.  Push and count: |gpu - oracle| <= 1e-4 oracle(|v|), as on the
    other routes."""
    from nitorch_amd import grid as G
    rng = np.random.default_rng(order)
    shape = (102, 101, 103)
    g = np.stack(np.meshgrid(*[np.arange(n, dtype=np.float64) for n in shape], indexing="ij"), -1)[None]
    g = (g + rng.uniform(-0.6, 0.6, g.shape)).astype(np.float32)
    far = rng.random(g.shape[:-1]) < 0.02
    g[far, rng.integers(0, 3, far.sum())] = rng.choice([3e9, 1e10, -1e10, np.inf, -np.inf], far.sum())
    g64 = np.nan_to_num(g.astype(np.float64), posinf=1e10, neginf=-1e10)
    x = rng.standard_normal((1, 3) + shape).astype(np.float32)
    x64 = x.astype(np.float64)
    if order > 1:   # (at order 1, three channels are read straight from the caches)
        pull = G.grid_pull(T(x), T(g), ["zero"], [order], 1)
        assert close(pull, O.grid_pull(x64, g64, "zero", order, 1, oob_f32=True))
        grad = G.grid_grad(T(x), T(g), ["zero"], [order], 1)
        assert close(grad, O.grid_grad(x64, g64, "zero", order, 1, oob_f32=True))
    push = G.grid_push(T(x), T(g), list(shape), ["zero"], [order], 1).cpu().double().numpy()
    bar = O.grid_push(np.abs(x64), g64, shape, "zero", order, 1, oob_f32=True)
    assert (np.abs(push - O.grid_push(x64, g64, shape, "zero", order, 1, oob_f32=True)) <= 1e-4 * bar + 1e-36).all()
    count = G.grid_count(T(g), list(shape), ["zero"], [order], 1).cpu().double().numpy()
    ref = O.grid_count(g64, shape, "zero", order, 1, oob_f32=True)
    assert (np.abs(count - ref) <= 1e-4 * ref + 1e-36).all()


@pytest.mark.parametrize("order", [0, 1, 2, 3, 5, 7])
@pytest.mark.parametrize("channels", [1, 4])
def test_infinite_coordinates_read_as_zero(order, channels):
    """Under `zero`, samples beyond the integer range or infinite along an
    axis read as zero whatever their weights (infinite or NaN there), alone
    in their tile and as whole tiles."""
    from nitorch_amd import grid as G
    rng = np.random.default_rng(10 * order + channels)
    shape, source = (8, 8, 48), (9, 10, 50)
    g = np.stack(np.meshgrid(*[np.arange(n, dtype=np.float64) for n in shape], indexing="ij"), -1)[None]
    g = (g + rng.uniform(-0.6, 0.6, g.shape)).astype(np.float32)
    values = [3e9, 1e10, -1e10, 1e30, np.inf, -np.inf]
    g[0, 1, 2, 16:32] = np.inf
    g[0, 1:3, 3, 5, 1] = -np.inf
    g[0, 4, 4, 16:20, 2] = 1e10
    for k, v in enumerate(values):   # whole tiles of 4 x 8 x 16
        h = g.copy()
        h[0, :4, :, 32:, k % 3] = v
        h[0, 4:, :, :16] = v
        h64 = np.nan_to_num(h.astype(np.float64), posinf=1e10, neginf=-1e10).clip(-1e10, 1e10)
        x = rng.standard_normal((1, channels) + source).astype(np.float32)
        u = rng.standard_normal((1, channels) + shape).astype(np.float32)
        x64, u64 = x.astype(np.float64), u.astype(np.float64)
        pull = G.grid_pull(T(x), T(h), ["zero"], [order], 1)
        assert close(pull, O.grid_pull(x64, h64, "zero", order, 1, oob_f32=True)), v
        if order == 0:
            continue
        grad = G.grid_grad(T(x), T(h), ["zero"], [order], 1)
        assert close(grad, O.grid_grad(x64, h64, "zero", order, 1, oob_f32=True)), v
        ggrad, = G.grid_pull_backward(T(u), T(x), T(h).requires_grad_(), ["zero"], [order], 1)
        assert close(ggrad, O.grid_pull_backward(u64, x64, h64, "zero", order, 1, oob_f32=True)[1]), v


@pytest.mark.parametrize("order", [0, 1, 2, 3, 5])
@pytest.mark.parametrize("channels", [1, 4])
@pytest.mark.parametrize("flip", [(4,), (3,), (2,), (3, 4), (1, 2, 3, 4)])
def test_flipped_source_views(order, channels, flip):
    """A source whose strides are negative along some dims reads as its
    flipped copy, bit for bit; most tiles of 4 x 8 x 16 lie well inside it."""
    from nitorch_amd import _lib as L
    from nitorch_amd import grid as G
    rng = np.random.default_rng(order)
    shape, source = (8, 16, 32), (20, 28, 44)
    g = np.stack(np.meshgrid(*[np.arange(n, dtype=np.float64) for n in shape], indexing="ij"), -1)[None]
    g = T((g + 6 + rng.uniform(-0.6, 0.6, g.shape)).astype(np.float32))
    x = T(rng.standard_normal((1, channels) + source).astype(np.float32))
    strides = list(x.stride())
    first = sum((x.shape[d] - 1) * strides[d] for d in flip)
    view = [-s if d in flip else s for d, s in enumerate(strides)]
    b, o = L.i32arr([2] * 3), L.i32arr([order] * 3)
    for name, ref in (("grid_pull", G.grid_pull), ("grid_grad", G.grid_grad)):
        ref = ref(x.flip(flip), g, ["dct2"], [order], 0)
        out = torch.full_like(ref, 7.0)
        L.check(getattr(L.lib(), "ni_" + name)(
            L.dtype_code(x.dtype), 3, b, o, 0, 1, channels, L.i64arr(source), L.i64arr(shape),
            ctypes.c_void_p(x.data_ptr() + 4 * first), L.i64arr(view), L.ptr(g), L.strides(g), L.ptr(out),
            L.strides(out), L.stream_of(g)), name)
        assert torch.equal(out, ref), name
