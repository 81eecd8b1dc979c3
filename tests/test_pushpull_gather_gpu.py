"""GPU parity of the gathers (pull, grid_grad, the pull's grid gradient)
against the FP64 oracle where their dispatch and their boxes change: channel
counts on both sides of the cache / tile choice and of a partial channel
chunk, tiles whose box needs four, two or one channel a stage or does not
fit at all, lattices one off the 4 x 4 x 16 and 4 x 8 x 16 blocks, axes
shorter than the taps, and sources whose z stride is not 1.

Tolerances: 1e-5 norm-relative (float sums of at most (order + 1)^3 terms,
(5 + 1)^3 ulps = 2.6e-5 at worst, a tenth of it in practice); order 0 exact.
"""
import numpy as np
import pytest
import torch

from oracle import pushpull as O

pytestmark = pytest.mark.gpu


def T(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def grid(rng, shape, source, kind):
    g = np.stack(np.meshgrid(*[np.linspace(0, s - 1, n) for n, s in zip(shape, source)], indexing="ij"), -1)[None]
    if kind == "stretch":       # neighbouring samples several voxels apart: wide boxes
        g = (g - np.array(source) / 2) * 2.5 + np.array(source) / 2
    elif kind == "scatter":     # no box holds a tile
        g = rng.uniform(-3, np.array(source) + 2, g.shape)
    g = g + rng.uniform(-0.6, 0.6, g.shape)
    return g.astype(np.float32)


def check(a, b, order, what):
    a = a.detach().cpu().double().numpy()
    if order == 0:
        assert np.array_equal(a, b), what
    assert np.abs(a - b).max() <= 1e-5 * max(np.abs(b).max(), 1e-30), what


@pytest.mark.parametrize("order", [0, 1, 2, 3, 5, 7])
@pytest.mark.parametrize("channels", [1, 2, 3, 4, 5])
def test_gather_paths(order, channels):
    from nitorch_amd import grid as G
    rng = np.random.default_rng(100 * order + channels)
    shapes = [((5, 9, 17), (5, 9, 17)), ((4, 8, 16), (37, 23, 41)), ((9, 7, 33), (40, 30, 50)), ((6, 5, 4), (3, 2, 4))]
    for (shape, source), kind in zip(shapes, ("near", "stretch", "scatter", "near")):
        g = grid(rng, shape, source, kind)
        x = rng.standard_normal((1, channels) + source).astype(np.float32)
        d = rng.standard_normal((1, channels) + shape).astype(np.float32)
        g64, x64, d64 = (t.astype(np.float64) for t in (g, x, d))
        for bound in ("dct2", "dst1", "dft", "zero"):
            for extrap in (0, 1):
                case = (kind, order, channels, bound, extrap)
                # channels last: the source's z stride is the channel count
                for xt in (T(x), T(np.moveaxis(x, 1, -1)).movedim(-1, 1)):
                    out = G.grid_pull(xt, T(g), [bound], [order], extrap)
                    check(out, O.grid_pull(x64, g64, bound, order, extrap, oob_f32=True), order, ("pull",) + case)
                    if order == 0:
                        continue
                    out = G.grid_grad(xt, T(g), [bound], [order], extrap)
                    check(out, O.grid_grad(x64, g64, bound, order, extrap, oob_f32=True), order, ("grad",) + case)
                    gt = T(g).requires_grad_()
                    out, = G.grid_pull_backward(T(d), xt, gt, [bound], [order], extrap)
                    ref = O.grid_pull_backward(d64, x64, g64, bound, order, extrap, oob_f32=True)[1]
                    check(out, ref, order, ("grid gradient",) + case)


@pytest.mark.parametrize("order", [1, 2, 3])
@pytest.mark.parametrize("channels", [1, 4])
def test_outside_taps_are_not_read(order, channels):
    """Under `zero`, a sample's taps outside the source read as zero whatever
    the voxel they fold to holds; a NaN reaches only the samples whose own
    taps touch it."""
    from nitorch_amd import grid as G
    rng = np.random.default_rng(order)
    shape = (9, 10, 18)
    g = grid(rng, shape, shape, "near")
    x = rng.standard_normal((1, channels) + shape).astype(np.float32)
    x[:, :, 0, 0, 0] = np.nan
    out = G.grid_pull(T(x), T(g), ["zero"], [order], 1).cpu().numpy()
    ref = O.grid_pull(x.astype(np.float64), g.astype(np.float64), "zero", order, 1, oob_f32=True)
    assert np.isnan(ref).any() and np.array_equal(np.isnan(out), np.isnan(ref))


@pytest.mark.parametrize("order", [1, 2, 3])
@pytest.mark.parametrize("channels", [8, 9])
def test_wide_channels_last_sources(order, channels):
    """Sources of eight channels and more whose z stride is not 1: boxes that
    would stage few channels at a time are read from the caches (order 1) or
    sorted into bins (2^20 samples and more).  Small calls against the
    oracle; large ones against the contiguous source."""
    from nitorch_amd import grid as G
    rng = np.random.default_rng(300 + 10 * order + channels)
    for kind in ("near", "stretch", "scatter"):
        shape, source = (5, 9, 33), (37, 23, 41)
        g = grid(rng, shape, source, kind)
        x = rng.standard_normal((1, channels) + source).astype(np.float32)
        d = rng.standard_normal((1, channels) + shape).astype(np.float32)
        g64, x64, d64 = (t.astype(np.float64) for t in (g, x, d))
        xt = T(np.moveaxis(x, 1, -1)).movedim(-1, 1)
        for bound, extrap in (("dct2", 0), ("zero", 1)):
            case = (kind, order, channels, bound, extrap)
            out = G.grid_pull(xt, T(g), [bound], [order], extrap)
            check(out, O.grid_pull(x64, g64, bound, order, extrap, oob_f32=True), order, ("pull",) + case)
            out = G.grid_grad(xt, T(g), [bound], [order], extrap)
            check(out, O.grid_grad(x64, g64, bound, order, extrap, oob_f32=True), order, ("grad",) + case)
            out, = G.grid_pull_backward(T(d), xt, T(g).requires_grad_(), [bound], [order], extrap)
            ref = O.grid_pull_backward(d64, x64, g64, bound, order, extrap, oob_f32=True)[1]
            check(out, ref, order, ("grid gradient",) + case)
        g = grid(rng, (102, 101, 103), (102, 101, 103), kind)
        x = torch.from_numpy(rng.standard_normal((1, 102, 101, 103, channels)).astype(np.float32)).cuda().movedim(-1, 1)
        for fn in (G.grid_pull, G.grid_grad):
            ref = fn(x.contiguous(), T(g), ["dct2"], [order], 0).cpu().double().numpy()
            check(fn(x, T(g), ["dct2"], [order], 0), ref, order, (fn.__name__, kind))


@pytest.mark.parametrize("channels", [1, 3, 9])
def test_nearest_grid_gradient_is_zero(channels):
    """Whatever the source holds: nothing of it is read."""
    from nitorch_amd import grid as G
    rng = np.random.default_rng(channels)
    shape = (5, 9, 17)
    g = T(grid(rng, shape, shape, "near")).requires_grad_()
    x = torch.full((1, channels) + shape, float("nan"), device="cuda")
    out, = G.grid_pull_backward(torch.ones_like(x), x, g, ["dct2"], [0], 1)
    assert out.shape == g.shape and not out.any()


@pytest.mark.parametrize("shape", [(150, 1, 1), (1, 150, 1), (1, 1, 150), (33, 21, 1), (21, 33, 2), (9, 16, 3), (9, 15, 3),
                                   (21, 1, 33)])
@pytest.mark.parametrize("channels", [1, 4])
def test_thin_lattices(shape, channels):
    """Points, slices and a few slices, whose axes the gathers relabel."""
    from nitorch_amd import grid as G
    rng = np.random.default_rng(400 + channels)
    source = (17, 23, 19)
    x = rng.standard_normal((2, channels) + source).astype(np.float32)
    d = rng.standard_normal((2, channels) + shape).astype(np.float32)
    for kind in ("near", "scatter"):
        g = np.concatenate([grid(rng, shape, source, kind) for _ in range(2)])
        g64, x64, d64 = (t.astype(np.float64) for t in (g, x, d))
        # the grid's components apart, the upstream channels last
        gt = T(np.moveaxis(g, -1, 1)).movedim(1, -1)
        dt = T(np.moveaxis(d, 1, -1)).movedim(-1, 1)
        for order in (1, 2, 3):
            case = (shape, channels, kind, order)
            out = G.grid_pull(T(x), gt, ["dct2"], [order], 0)
            check(out, O.grid_pull(x64, g64, "dct2", order, 0, oob_f32=True), order, ("pull",) + case)
            out = G.grid_grad(T(x), gt, ["dct2"], [order], 0)
            check(out, O.grid_grad(x64, g64, "dct2", order, 0, oob_f32=True), order, ("grad",) + case)
            out, = G.grid_pull_backward(dt, T(x), gt.clone().requires_grad_(), ["dct2"], [order], 0)
            ref = O.grid_pull_backward(d64, x64, g64, "dct2", order, 0, oob_f32=True)[1]
            check(out, ref, order, ("grid gradient",) + case)
