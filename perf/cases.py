"""Performance cases of the framework: the calls that programs built on it make.

Each case is one pass through a public entry point, on inputs made on the GPU
from a seed:

  pull / push / grad   `spatial.grid_pull / grid_push / grid_grad`: sampling,
                       splatting and spatial gradients of images on a grid
  train                `spatial.grid_pull` and its backward for both inputs
  reslice              `spatial.reslice`: prefilter, then a pull through an
                       affine map
  resize               `resize.resize`: edge-aligned resize by a factor
  fmg                  `solve.solve_grid_fmg`: one full multigrid pass on a
                       Gauss-Newton system of a displacement field
  svf                  `svf.exp` with the analytic backward: integration of a
                       stationary velocity and of its gradient
  unet                 `learned.UNet.pack` + `forward`: the learned
                       preconditioner's network

Grids come in three kinds: "near" (the benchmark's recipe: the identity plus
a small smooth displacement, 5 % of the points moved out of bounds), "warp"
(a smooth displacement of `std` voxels RMS) and "affine" (a rotation and a
zoom about the centre).

`exact` restates every path but the multigrid iterate in plain float64 torch.
"""
import math

import torch

DEVICE = "cuda"
OOB_TOL = 0.05
PENALTY = dict(absolute=1e-4, membrane=1e-3, bending=0.2, lame=(0.05, 0.2))


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # the smallest call in regular use: one coarse image, linear, where launches count
        dict(name="pull_96_o1", op="pull", N=1, C=1, X=96, Y=96, Z=96, order=1, bound="dct2", grid="warp", std=0.5),
        # the benchmark's workload: cubic pull and its adjoint on a large batch of feature volumes
        dict(name="pull_192_o3", op="pull", N=4, C=8, X=192, Y=192, Z=192, order=3, bound="dct2", grid="near", std=8.0),
        dict(name="push_192_o3", op="push", N=4, C=8, X=192, Y=192, Z=192, order=3, bound="dct2", grid="near", std=8.0),
        # tissue classes splatted into template space through a strong nonlinear warp; ragged brain-sized lattice
        dict(name="push_warp_o1", op="push", N=1, C=4, X=181, Y=217, Z=181, order=1, bound="dct2", grid="warp", std=8.0),
        # gradients of the moving image in a registration's Gauss-Newton step
        dict(name="grad_warp_o1", op="grad", N=1, C=1, X=160, Y=192, Z=160, order=1, bound="dft", grid="warp", std=4.0),
        # a spatial-transformer layer in training: forward and both gradients
        dict(name="train_128_o3", op="train", N=2, C=3, X=128, Y=160, Z=128, order=3, bound="dft", grid="near", std=8.0),
        # one image resliced into a rotated, zoomed space, cubic with prefilter
        dict(name="reslice_181_o3", op="reslice", N=1, C=1, X=181, Y=217, Z=181, order=3, bound="dct2", angle=15.0,
             zoom=1.1),
        # one level of an image pyramid
        dict(name="resize_half_o3", op="resize", N=4, C=8, X=192, Y=192, Z=192, order=3, bound="dct2", factor=0.5),
        # the Gauss-Newton step of a whole-brain registration, default smoother
        dict(name="fmg_160_cg", op="fmg", N=1, X=160, Y=192, Z=160, bound="dft", optim="cg", nb_iter=4),
        # the same on a coarse, ragged lattice with the Gauss-Seidel smoother: latency
        dict(name="fmg_63_relax", op="fmg", N=1, X=63, Y=77, Z=58, bound="dct2", optim="relax", nb_iter=2),
        # integration of a velocity field and of its gradient in a diffeomorphic registration
        dict(name="svf_160", op="svf", N=1, X=160, Y=192, Z=160, steps=8, vmax=3.0),
        # one application of the learned preconditioner
        dict(name="unet_160", op="unet", N=1, X=160, Y=192, Z=160),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _edges(rng, lo, hi):
    """Three edges of a lattice within 30 % of a common size: volumes are roughly cubic."""
    base = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return [max(lo, min(hi, int(round(base * rng.uniform(0.8, 1.2))))) for _ in range(3)]


def draw(rng):
    op = rng.choice(["pull", "pull", "push", "push", "grad", "train", "reslice", "resize", "fmg", "svf", "unet"])
    bound = rng.choice(["dct2", "dft", "replicate", "zero"])
    if op in ("pull", "push", "grad", "train"):
        X, Y, Z = _edges(rng, 48, 192)
        order = rng.choice([1, 1, 2, 3, 3, 5]) if op != "train" else rng.choice([1, 3])
        N, C = rng.choice([1, 1, 2, 4]), rng.choice([1, 1, 2, 3, 4, 8] if op != "grad" else [1, 1, 2, 4])
        grid = rng.choice(["near", "warp", "warp", "affine"])
        case = dict(op=op, N=N, C=C, X=X, Y=Y, Z=Z, order=order, bound=bound, grid=grid)
        if grid == "affine":
            return dict(case, angle=round(rng.uniform(2, 30), 1), zoom=round(rng.uniform(0.8, 1.25), 2))
        return dict(case, std=8.0 if grid == "near" else round(rng.uniform(0.5, 8.0), 1))
    if op == "reslice":
        X, Y, Z = _edges(rng, 48, 217)
        return dict(op=op, N=1, C=rng.choice([1, 1, 3]), X=X, Y=Y, Z=Z, order=rng.choice([1, 3, 3]),
                    bound=rng.choice(["dct2", "dft"]), angle=round(rng.uniform(2, 30), 1),
                    zoom=round(rng.uniform(0.8, 1.25), 2))
    if op == "resize":
        factor = rng.choice([0.5, 0.5, 2.0])
        X, Y, Z = _edges(rng, 48, 192 if factor < 1 else 120)
        return dict(op=op, N=rng.choice([1, 2, 4]), C=rng.choice([1, 3, 8]), X=X, Y=Y, Z=Z,
                    order=rng.choice([1, 3, 3]), bound=rng.choice(["dct2", "dft"]), factor=factor)
    if op == "fmg":
        X, Y, Z = _edges(rng, 32, 176)
        return dict(op=op, N=1, X=X, Y=Y, Z=Z, bound=rng.choice(["dft", "dct2"]), optim=rng.choice(["cg", "cg", "relax"]),
                    nb_iter=rng.choice([2, 4]))
    if op == "svf":
        X, Y, Z = _edges(rng, 48, 176)
        return dict(op=op, N=1, X=X, Y=Y, Z=Z, steps=rng.choice([6, 8]), vmax=round(rng.uniform(1.0, 4.0), 1))
    X, Y, Z = (4 * (e // 4) for e in _edges(rng, 32, 176))
    return dict(op=op, N=1, X=X, Y=Y, Z=Z)


# ----------------------------------------------------------------- the inputs
def _smooth(field, sigma):
    """Periodic Gaussian smoothing over the last three dims, one circulant product an axis."""
    for d in (-3, -2, -1):
        n = field.shape[d]
        i = torch.arange(n, device=field.device)
        gap = (i[:, None] - i[None]).remainder(n)
        gap = torch.minimum(gap, n - gap).to(field.dtype)
        g = torch.exp(-0.5 * (gap / sigma) ** 2)
        g = g / g.sum(1, keepdim=True)
        field = torch.matmul(field.movedim(d, -1), g).movedim(-1, d)
    return field.contiguous()


def _identity(shape, dtype=torch.float32):
    mesh = torch.meshgrid(*[torch.arange(n, dtype=dtype, device=DEVICE) for n in shape], indexing="ij")
    return torch.stack(mesh, -1)


def _rotation(case):
    """Affine matrix (3, 4) of the case's rotation about y and zoom, about the centre of the lattice."""
    a = math.radians(case["angle"])
    rot = torch.tensor([[math.cos(a), 0.0, math.sin(a)], [0.0, 1.0, 0.0], [-math.sin(a), 0.0, math.cos(a)]],
                       dtype=torch.float64) * case["zoom"]
    centre = torch.tensor([(case[k] - 1) / 2 for k in "XYZ"], dtype=torch.float64)
    return torch.cat([rot, (centre - rot @ centre)[:, None]], 1)


def _grid(case, gen):
    """Sampling grid (N, X, Y, Z, 3) of the case, in voxels."""
    N, shape = case["N"], (case["X"], case["Y"], case["Z"])
    if case["grid"] == "affine":
        mat = _rotation(case).to(DEVICE)
        out = _identity(shape, torch.float64) @ mat[:, :3].T + mat[:, 3]
        return out.float().expand(N, *out.shape).contiguous()
    noise = torch.randn((N, 3) + shape, generator=gen, device=DEVICE)
    disp = _smooth(noise, 10.0) * case["std"]
    if case["grid"] == "warp":
        disp *= case["std"] / disp.std()
    out = _identity(shape) + disp.movedim(1, -1)
    if case["grid"] == "near":
        lattice = out.shape[:-1]
        moved = torch.rand(lattice, generator=gen, device=DEVICE) < 0.05
        axis = torch.randint(3, lattice, generator=gen, device=DEVICE)
        sign = torch.randint(2, lattice, generator=gen, device=DEVICE) * 2 - 1
        for d in range(3):
            out[..., d] += (moved & (axis == d)) * sign * float(shape[d])
    return out.contiguous()


def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _image(case, gen):
    return torch.rand((case["N"], case["C"], case["X"], case["Y"], case["Z"]), generator=gen, device=DEVICE)


def _system(case, gen):
    """Hessian (N, *shape, 6) and gradient (N, *shape, 3) of a Gauss-Newton step."""
    lattice = (case["N"], case["X"], case["Y"], case["Z"])
    g = _smooth(torch.randn((lattice[0], 3) + lattice[1:], generator=gen, device=DEVICE), 2.0)
    diag = torch.rand(lattice + (3,), generator=gen, device=DEVICE) * 1.5 + 0.5
    off = torch.rand(lattice + (3,), generator=gen, device=DEVICE) * 0.4 - 0.2
    return torch.cat([diag, off], -1), (g / g.std()).movedim(1, -1).contiguous()


def prepare(case, seed):
    gen = _generator(seed)
    op = case["op"]
    state = {"case": case}
    if op in ("pull", "push", "grad", "train"):
        state["grid"] = _grid(case, gen)
        state["image"] = _image(case, gen)
        if op == "train":
            state["grid"].requires_grad_(True)
            state["image"].requires_grad_(True)
            state["upstream"] = torch.randn(state["image"].shape, generator=gen, device=DEVICE)
    elif op == "reslice":
        state["image"] = _image(case, gen)[0]
        # orientation matrices of the image and of the target lattice
        bottom = torch.tensor([[0.0, 0.0, 0.0, 1.0]])
        state["affine"] = torch.eye(4, device=DEVICE)
        state["affine_to"] = torch.cat([_rotation(case).float(), bottom]).to(DEVICE)
    elif op == "resize":
        state["image"] = _image(case, gen)
    elif op == "fmg":
        state["hessian"], state["gradient"] = _system(case, gen)
    elif op == "svf":
        lattice = (case["X"], case["Y"], case["Z"])
        v = _smooth(torch.randn((case["N"], 3) + lattice, generator=gen, device=DEVICE), 4.0)
        state["velocity"] = (v * (case["vmax"] / v.abs().max())).movedim(1, -1).contiguous().requires_grad_(True)
        state["upstream"] = torch.randn((case["N"],) + lattice + (3,), generator=gen, device=DEVICE)
    elif op == "unet":
        from nitorch_amd import learned
        state["net"] = learned.UNet.load(learned.default_weights_path(), DEVICE)
        h, g = _system(case, gen)
        state["hessian"], state["gradient"] = (t.movedim(-1, 1).contiguous() for t in (h, g))
    return state


# ------------------------------------------------------------------- the pass
def run(state):
    case = state["case"]
    op = case["op"]
    if op in ("pull", "push", "grad", "train"):
        from nitorch_amd import spatial
        opt = dict(interpolation=case["order"], bound=case["bound"], extrapolate=False)
        if op == "pull":
            return spatial.grid_pull(state["image"], state["grid"], **opt)
        if op == "push":
            return spatial.grid_push(state["image"], state["grid"], **opt)
        if op == "grad":
            return spatial.grid_grad(state["image"], state["grid"], **opt)
        out = spatial.grid_pull(state["image"], state["grid"], **opt)
        d_image, d_grid = torch.autograd.grad(out, (state["image"], state["grid"]), state["upstream"])
        return [out.detach(), d_image, d_grid]
    if op == "reslice":
        from nitorch_amd import spatial
        return spatial.reslice(state["image"], state["affine"], state["affine_to"], interpolation=case["order"],
                               bound=case["bound"])
    if op == "resize":
        from nitorch_amd import resize
        return resize.resize(state["image"], None, [case["factor"]], [case["bound"]], [case["order"]], ["edge"])
    if op == "fmg":
        from nitorch_amd import solve
        return solve.solve_grid_fmg(state["hessian"], state["gradient"], bound=case["bound"], optim=case["optim"],
                                    nb_cycles=2, nb_iter=case["nb_iter"], **PENALTY)
    if op == "svf":
        from nitorch_amd import svf
        out = svf.exp(state["velocity"], steps=case["steps"], anagrad=True)
        d_vel, = torch.autograd.grad(out, state["velocity"], state["upstream"])
        return [out.detach(), d_vel]
    net = state["net"]
    return net.forward(net.pack(state["gradient"], state["hessian"]))


# ----------------------------------------------------------------- its floors
def work(case):
    """Compulsory bytes (each input read once, each output written once) and operations of one pass."""
    op = case["op"]
    V = case["N"] * case["X"] * case["Y"] * case["Z"]
    if op in ("pull", "push", "grad", "train"):
        C, taps = case["C"], (case["order"] + 1) ** 3
        if op == "grad":
            return {"bytes": 4 * V * (3 + C + 3 * C), "flops": 6 * V * C * taps}
        if op == "train":   # forward, then the pushed gradient and the grid's gradient
            return {"bytes": 4 * V * ((3 + 2 * C) + (6 + 3 * C)), "flops": 10 * V * C * taps}
        return {"bytes": 4 * V * (3 + 2 * C), "flops": 2 * V * C * taps}
    if op == "reslice":
        C, o = case["C"], case["order"]
        # image in, result out; the filter's two recursions along three axes and the taps
        return {"bytes": 8 * V * C, "flops": V * C * (2 * (o + 1) ** 3 + (12 if o > 1 else 0)) + 18 * V}
    if op == "resize":
        C, f = case["C"], case["factor"]
        out = case["N"] * int(case["X"] * f) * int(case["Y"] * f) * int(case["Z"] * f)
        return {"bytes": 4 * C * (V + out), "flops": 2 * C * out * 3 * (case["order"] + 1)}
    if op == "fmg":
        # smoothing steps on the finest level: 2 cycles, before and after; 1/7 more on the coarser ones.  A step
        # reads the Hessian, the gradient (or residual) and the iterate, and writes the iterate
        steps = 2 * 2 * case["nb_iter"] * 8 / 7
        return {"bytes": 4 * V * (6 + 3 + 3 + 3) * steps, "flops": V * (2 * 3 * 25 + 2 * 15 + 40) * steps}
    if op == "svf":
        # a squaring reads and writes the velocity (forward, and twice again backward: with the gradient and the
        # Jacobian, which the analytic backward pushes along)
        s = case["steps"]
        return {"bytes": 4 * V * s * (6 + (3 + 9 + 3 + 12) * 2), "flops": V * s * 8 * 2 * (3 + 3 + 12)}
    taps = {"full": [(16, 16)] * 3 + [(48, 16), (16, 3)], "half": [(16, 32), (32, 32), (96, 32), (32, 32)],
            "quarter": [(32, 64), (64, 64)]}
    flops = sum(2 * 27 * ci * co * V // {"full": 1, "half": 8, "quarter": 64}[k] for k, v in taps.items() for ci, co in v)
    return {"bytes": 4 * V * (3 + 6 + 3), "flops": flops}


# ------------------------------------------------- the results, in 64 bits
def _spline(d, order):
    """B-spline of degree `order` (>= 0) at signed distance d: truncated powers."""
    half = (order + 1) / 2
    if order == 0:
        return ((d >= -half) & (d < half)).to(d.dtype)
    a = half - d.abs()
    out = torch.zeros_like(d)
    for k in range(int(half) + 1):
        out += (-1) ** k * math.comb(order + 1, k) * (a - k).clamp(min=0) ** order
    return out / math.factorial(order)


def _dspline(d, order):
    return _spline(d + 0.5, order - 1) - _spline(d - 0.5, order - 1)


def _fold(i, n, bound):
    """Index and validity of voxel i under a boundary condition."""
    one = torch.ones_like(i, dtype=torch.float64)
    if bound == "dft":
        return i.remainder(n), one
    if bound == "dct2":
        j = i.remainder(2 * n)
        return torch.where(j >= n, 2 * n - 1 - j, j), one
    if bound == "replicate":
        return i.clamp(0, n - 1), one
    return i.clamp(0, n - 1), ((i >= 0) & (i < n)).double()


def _taps(grid, shape, order, bound):
    """Yields (flat index, weight, d weight / d x, y, z) of every tap of the samples grid (S, 3); out-of-bound
    samples have zero weights unless `bound` is a pair (bound, True): extrapolated."""
    bound, extrapolate = bound if isinstance(bound, tuple) else (bound, False)
    size = torch.tensor(shape, device=grid.device, dtype=grid.dtype)
    inside = torch.ones(grid.shape[0], dtype=torch.bool, device=grid.device)
    if not extrapolate:
        inside = ((grid >= -OOB_TOL) & (grid < size - 1 + OOB_TOL)).all(-1)
    x = torch.where(inside[:, None], grid, torch.zeros_like(grid)).double()
    axes = []
    for d in range(3):
        lo = torch.floor(x[:, d] - (order - 1) / 2).long()
        axis = []
        for t in range(order + 1):
            j, ok = _fold(lo + t, shape[d], bound)
            dist = x[:, d] - (lo + t)
            axis.append((j, _spline(dist, order) * ok, _dspline(dist, order) * ok))
        axes.append(axis)
    inside = inside.double()
    for jx, wx, gx in axes[0]:
        for jy, wy, gy in axes[1]:
            wxy, jxy = wx * wy * inside, (jx * shape[1] + jy) * shape[2]
            gxy, hxy = gx * wy * inside, wx * gy * inside
            for jz, wz, gz in axes[2]:
                yield jxy + jz, wxy * wz, (gxy * wz, hxy * wz, wxy * gz)


CHUNK = 1 << 22   # samples a step of the float64 restatements handles at once


def _pull64(image, grid, order, bound):
    """(N, C, *shape) image at the (N, *out, 3) grid -> (N, C, *out), float64."""
    N, C, *shape = image.shape
    flat = image.double().reshape(N, C, -1).movedim(1, 2).contiguous()
    out = torch.zeros((N, grid[0, ..., 0].numel(), C), dtype=torch.float64, device=image.device)
    for n in range(N):
        for g, o in zip(grid[n].reshape(-1, 3).split(CHUNK), out[n].split(CHUNK)):
            for at, w, _ in _taps(g, shape, order, bound):
                o += flat[n][at] * w[:, None]
    return out.movedim(2, 1).reshape((N, C) + tuple(grid.shape[1:-1]))


def _push64(image, grid, order, bound):
    N, C, *shape = image.shape
    flat = image.double().reshape(N, C, -1).movedim(1, 2).contiguous()
    out = torch.zeros_like(flat)
    for n in range(N):
        for g, v in zip(grid[n].reshape(-1, 3).split(CHUNK), flat[n].split(CHUNK)):
            for at, w, _ in _taps(g, shape, order, bound):
                out[n].index_add_(0, at, v * w[:, None])
    return out.movedim(2, 1).reshape(image.shape)


def _grad64(image, grid, order, bound):
    N, C, *shape = image.shape
    flat = image.double().reshape(N, C, -1).movedim(1, 2).contiguous()
    out = torch.zeros((N, grid[0, ..., 0].numel(), C, 3), dtype=torch.float64, device=image.device)
    for n in range(N):
        for g, o in zip(grid[n].reshape(-1, 3).split(CHUNK), out[n].split(CHUNK)):
            for at, _, dw in _taps(g, shape, order, bound):
                o += flat[n][at][..., None] * torch.stack(dw, -1)[:, None]
    return out.movedim(2, 1).reshape((N, C) + tuple(grid.shape[1:-1]) + (3,))


def _along(mats, image):
    """Applies one matrix to each of the last three dims."""
    for d, m in zip((-3, -2, -1), mats):
        image = torch.matmul(image.movedim(d, -1), m.T).movedim(-1, d)
    return image


def _sampling_matrix(x, n, order, bound):
    """Matrix that samples a line of n spline coefficients at the coordinates x."""
    lo = torch.floor(x - (order - 1) / 2).long()
    m = torch.zeros((x.numel(), n), dtype=torch.float64, device=x.device)
    row = torch.arange(x.numel(), device=x.device)
    for t in range(order + 1):
        j, ok = _fold(lo + t, n, bound)
        m.index_put_((row, j), _spline(x - (lo + t), order) * ok, accumulate=True)
    return m


def _prefilter64(image, order, bound):
    if order < 2:
        return image.double()
    lines = [torch.arange(n, dtype=torch.float64, device=image.device) for n in image.shape[-3:]]
    return _along([torch.linalg.inv(_sampling_matrix(x, x.numel(), order, bound)) for x in lines], image.double())


def _jacobian64(disp):
    """I + central differences (periodic) of a (N, X, Y, Z, 3) displacement: [..., i, j] = d psi_i / d x_j."""
    parts = [(disp.roll(-1, d) - disp.roll(1, d)) / 2 for d in (1, 2, 3)]
    return torch.stack(parts, -1) + torch.eye(3, dtype=disp.dtype, device=disp.device)


def _at(field, grid):
    """A (N, X, Y, Z, K) field pulled linearly, periodic, at the grid."""
    return _pull64(field.movedim(-1, 1), grid, 1, ("dft", True)).movedim(1, -1)


def _svf64(velocity, upstream, steps):
    def compose(jac, grid, disp):
        left = _jacobian64(disp)
        return _at(left.flatten(-2), grid).reshape(left.shape) @ jac

    ident = _identity(velocity.shape[1:4], torch.float64)
    v = velocity.detach().double() / 2 ** steps
    jac = torch.eye(3, dtype=torch.float64, device=v.device).expand(v.shape + (3,))
    for _ in range(steps):
        grid = ident + v
        jac = compose(jac, grid, v)
        v = v + _at(v, grid)
    out = v + ident
    grad = (jac.transpose(-1, -2) @ upstream.double()[..., None])[..., 0]
    v = -velocity.detach().double() / 2 ** steps
    jac = _jacobian64(v)
    eye = torch.eye(3, dtype=torch.float64, device=v.device)
    grad = torch.linalg.solve_ex((2 * eye - jac).transpose(-1, -2), grad[..., None])[0][..., 0]
    for _ in range(steps):
        grid = ident + v
        pushed = (jac.transpose(-1, -2) @ _at(grad, grid)[..., None])[..., 0]
        a, b, c = jac.unbind(-1)
        grad = grad + (torch.linalg.cross(a, b) * c).sum(-1, keepdim=True) * pushed
        jac = compose(jac, grid, v)
        v = v + _at(v, grid)
    return [out, grad / 2 ** steps]


def _conv64(x, net, name, act=True):
    """3 x 3 x 3 zero-padded convolution of a (X, Y, Z, CI) activation with the network's bf16 weights, one product
    a tap."""
    w = net.params[name + ".w"].to(torch.bfloat16).double()
    X, Y, Z = x.shape[:3]
    pad = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1, 1, 1))
    y = net.params[name + ".b"].double().expand(X, Y, Z, -1).clone()
    for t in range(27):
        i, j, k = t // 9, t // 3 % 3, t % 3
        part = pad[i:i + X, j:j + Y, k:k + Z, :w.shape[-1]]
        y += part @ w[:, i, j, k].T
    return torch.where(y > 0, y, 0.1 * y) if act else y


def _pool64(x):
    X, Y, Z, C = x.shape
    return x.reshape(X // 2, 2, Y // 2, 2, Z // 2, 2, C).mean((1, 3, 5))


def _up64(x):
    for d in range(3):
        x = x.repeat_interleave(2, d)
    return x


def _unet64(net, hessian, gradient):
    out = []
    for h, g in zip(hessian, gradient):
        x = torch.cat([g, h]).to(torch.bfloat16).double().movedim(0, -1)
        full = _conv64(_conv64(x, net, "e1a"), net, "e1b")
        half = _conv64(_conv64(_pool64(full), net, "e2a"), net, "e2b")
        deep = _conv64(_conv64(_pool64(half), net, "b1"), net, "b2")
        half = _conv64(_conv64(torch.cat([_up64(deep), half], -1), net, "d2a"), net, "d2b")
        full = _conv64(_conv64(torch.cat([_up64(half), full], -1), net, "d1a"), net, "d1b")
        out.append(_conv64(full, net, "head", act=False))
    return torch.stack(out)


def exact(case, seed):
    state = prepare(case, seed)
    op = case["op"]
    with torch.no_grad():
        if op == "fmg":      # an iterate of the solver, not the solution: no closed form
            return None
        if op in ("pull", "push", "grad"):
            fn = {"pull": _pull64, "push": _push64, "grad": _grad64}[op]
            return fn(state["image"], state["grid"], case["order"], case["bound"])
        if op == "train":
            image, grid, up = (state[k].detach() for k in ("image", "grid", "upstream"))
            d_grid = (_grad64(image, grid, case["order"], case["bound"]) * up.double()[..., None]).sum(1)
            return [_pull64(image, grid, case["order"], case["bound"]),
                    _push64(up, grid, case["order"], case["bound"]), d_grid]
        if op == "reslice":
            mat = state["affine_to"].double()
            grid = _identity(state["image"].shape[-3:], torch.float64) @ mat[:3, :3].T + mat[:3, 3]
            coeff = _prefilter64(state["image"], case["order"], case["bound"])
            return _pull64(coeff[None], grid[None], case["order"], case["bound"])[0]
        if op == "resize":
            mats = []
            for n in state["image"].shape[-3:]:
                m = int(n * case["factor"])
                x = torch.arange(m, dtype=torch.float64, device=DEVICE) * (n / m) + 0.5 * (n / m - 1)
                mats.append(_sampling_matrix(x, n, case["order"], case["bound"]))
            return _along(mats, state["image"].double())
        if op == "svf":
            return _svf64(state["velocity"], state["upstream"], case["steps"])
        return _unet64(state["net"], state["hessian"], state["gradient"])
