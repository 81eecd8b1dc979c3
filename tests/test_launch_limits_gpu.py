"""GPU checks of calls whose blocks, mostly idle, come to more than 2^32
work-items (which a launch counts in 32 bits): they take another kernel and
give what smaller calls or the general path give.  3 to 4 GB of inputs each."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_thin_pull():
    """2^25 rows of 8 samples, one z: 4 x 4 x 16 blocks, 2^24 of 256 threads."""
    from nitorch_amd import grid as G
    gen = torch.Generator(device="cuda").manual_seed(0)
    n = 2 ** 25
    x = torch.rand((1, 1, 16, 8, 1), generator=gen, device="cuda")
    g = torch.rand((1, n, 8, 1, 3), generator=gen, device="cuda") * torch.tensor([15.0, 7.0, 0.0], device="cuda")
    out = G.grid_pull(x, g, ["dct2"], [1], 0)
    for part in (slice(0, 1000), slice(n // 2 - 500, n // 2 + 500), slice(n - 1000, n)):
        ref = G.grid_pull(x, g[:, part].contiguous(), ["dct2"], [1], 0)
        assert (out[:, :, part] - ref).abs().max() <= 1e-6   # another order of eight products


def test_thin_push():
    """2^26 points in a row: 8 x 16 x 16 tiles, 2^23 of 512 threads."""
    from nitorch_amd import grid as G
    gen = torch.Generator(device="cuda").manual_seed(1)
    n = 2 ** 26
    g = torch.rand((1, n, 1, 1, 3), generator=gen, device="cuda") * torch.tensor([15.0, 7.0, 3.0], device="cuda")
    out = G.grid_count(g, [16, 8, 4], ["dct2"], [1], 1)
    # every point adds one in all; half a million sums of 2^-24 relative steps a voxel
    assert abs(out.double().sum().item() / n - 1) <= 1e-2
    half = G.grid_count(g[:, :n // 2].contiguous(), [16, 8, 4], ["dct2"], [1], 1)
    assert (out / half - 2).abs().max() <= 0.1


def test_many_small_velocities():
    """2^23 lattices of 4 x 4 x 2: 4 x 2 x 32 blocks, 2^24 of 256 threads."""
    from nitorch_amd import svf
    gen = torch.Generator(device="cuda").manual_seed(2)
    n = 2 ** 23
    v = torch.rand((n, 4, 4, 2, 3), generator=gen, device="cuda") - 0.5
    assert svf._fused(v, "linear", "dft") is None and svf._fused(v[:n - 1], "linear", "dft") is not None
    out = svf.exp_forward(v, steps=2)
    for part in (slice(0, 100), slice(n - 100, n)):
        ref = svf.exp_forward(v[part].contiguous(), steps=2)
        assert (out[part] - ref).abs().max() <= 2e-6   # a few roundings of 4


def test_many_small_resizes():
    """2^24 volumes of 4^3: a block each."""
    from nitorch_amd import resize as R
    gen = torch.Generator(device="cuda").manual_seed(3)
    x = torch.rand((2 ** 24, 1, 4, 4, 4), generator=gen, device="cuda")
    out = R.resize(x, None, [0.5], ["dct2"], [1], ["edge"])
    for part in (slice(0, 100), slice(2 ** 24 - 100, 2 ** 24)):
        ref = R.resize(x[part].contiguous(), None, [0.5], ["dct2"], [1], ["edge"])
        assert (out[part] - ref).abs().max() <= 1e-6
