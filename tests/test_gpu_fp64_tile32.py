"""GPU parity of the FP64 form on 32-point tiles (k_tile32_f64) against the FP64 direct-sweep oracle.

Bar: max|gpu - oracle| / max|oracle| <= 1e-12, as for the 16-point FP64 form.  The depths cover the
reduced inverse stages (valid width V = 32 - 2 r t <= 16, at the window offset of either index
convention) and the full ones, with tail blocks of another depth, and grids smaller than a tile.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL_FP64 = 1e-12


def _run(ffs, torch, x, radius, w, steps, **kw):
    plan = ffs.Plan(x.ndim, x.shape, w, radius, steps, **kw)
    d_in = torch.from_numpy(np.ascontiguousarray(x)).cuda()
    d_out = torch.empty_like(d_in)
    plan.run(d_in, d_out)
    torch.cuda.synchronize()
    info = plan.info
    plan.close()
    return d_out.cpu().numpy(), info


@pytest.mark.parametrize("shape", ["Heat-2D", "Box2D9P", "Star2D9P", "Box2D25P"])
@pytest.mark.parametrize("size", [(37, 53), (16, 16), (5, 7), (64, 40), (1, 19)])
@pytest.mark.parametrize("steps", [1, 4, 9, 17])
def test_2d_fp64_tile32_named(ffs, oracle, torch_cuda, shape, size, steps):
    _, r, w, _ = ffs.named_stencil(shape, seed=11)
    x = oracle.uniform(777 + size[0] * 31 + size[1], size)
    got, info = _run(ffs, torch_cuda, x, r, w, steps, tile=32)
    assert info["tile"][:2] == [32, 32]
    ref = oracle.sweep(x, r, w, steps)
    rel = oracle.errors(got, ref)[1]
    assert rel <= TOL_FP64, (shape, size, steps, info, rel)


@pytest.mark.parametrize("convention", ["ref", "centred"])
@pytest.mark.parametrize("radius,fuse", [(1, 7), (1, 8), (2, 3), (2, 4), (3, 2), (3, 3), (4, 2)])
def test_2d_fp64_tile32_depths(ffs, oracle, torch_cuda, convention, radius, fuse):
    rng = np.random.default_rng(10 * radius + fuse)
    w = rng.random((2 * radius + 1) ** 2)
    w /= w.sum()
    x = oracle.uniform(5 + fuse, (70, 45))
    steps = 2 * fuse + 1
    got, info = _run(ffs, torch_cuda, x, radius, w, steps, tile=32, fuse=fuse, convention=convention)
    assert info["valid"][0] == 32 - 2 * radius * fuse
    ref = oracle.sweep(x, radius, w, steps, convention=0 if convention == "ref" else 1)
    assert oracle.errors(got, ref)[1] <= TOL_FP64, (convention, radius, fuse, info)


def test_2d_fp64_tile32_matches_tile16_at_scale(ffs, torch_cuda):
    # 2048^2 x 16 steps: the two FP64 tile families agree to FP64 rounding (size-independent check)
    torch = torch_cuda
    _, r, w, _ = ffs.named_stencil("Box2D25P", seed=0x5EED0002)
    n = 2048
    d_in = torch.empty(n * n, dtype=torch.float64, device="cuda").reshape(n, n)
    ffs.fill_uniform_device(99, d_in)
    outs = []
    for tile in (16, 32):
        plan = ffs.Plan(2, (n, n), w, r, 16, tile=tile)
        d_out = torch.empty_like(d_in)
        plan.run(d_in, d_out)
        torch.cuda.synchronize()
        plan.close()
        outs.append(d_out)
    rel = float((outs[0] - outs[1]).abs().max() / outs[0].abs().max())
    assert rel <= TOL_FP64, rel


@pytest.mark.parametrize("n1", [1 << 22, (1 << 22) + 96])
@pytest.mark.parametrize("precision", ["fp64", "f16", "bf16"])
def test_2d_tile32_long_rows(ffs, oracle, torch_cuda, n1, precision):
    # Rows of 2^22 columns are the widest whose interior windows are read through the 32-bit buffer
    # offsets; wider rows take the general gather for every window.  Both agree with the oracle.
    _, r, w, _ = ffs.named_stencil("Heat-2D", seed=3)
    x = oracle.uniform(4242 + n1, (34, n1))
    got, info = _run(ffs, torch_cuda, x, r, w, 3, tile=32, precision=precision)
    assert info["tile"][:2] == [32, 32]
    ref = oracle.sweep(x, r, w, 3)
    tol = TOL_FP64 if precision == "fp64" else 1e-6
    assert oracle.errors(got, ref)[1] <= tol, (precision, n1, info)


@pytest.mark.parametrize("convention", ["ref", "centred"])
@pytest.mark.parametrize("radius,fuse,size", [(0, 3, (65, 31)), (15, 1, (9, 40)), (7, 1, (35, 37)), (5, 2, (25, 24)),
                                              (1, 15, (3, 130)), (2, 4, (17, 15)), (2, 4, (16, 272)), (1, 1, (31, 61))])
def test_2d_fp64_tile32_edges(ffs, oracle, torch_cuda, convention, radius, fuse, size):
    # The real half-sample transforms at the ends of their range: every position valid (V = 32), V = 2, V = 18
    # (one column past the reduced block), the widest shift of the filter (radius 15), signed taps, and
    # grids one short of, equal to and one past a tile.
    rng = np.random.default_rng(31 * radius + fuse)
    w = rng.standard_normal((2 * radius + 1) ** 2)
    w /= np.abs(w).sum()
    x = oracle.uniform(9 + radius, size)
    got, info = _run(ffs, torch_cuda, x, radius, w, fuse, tile=32, fuse=fuse, convention=convention)
    assert info["tile"][:2] == [32, 32] and info["valid"][0] == 32 - 2 * radius * fuse
    ref = oracle.sweep(x, radius, w, fuse, convention=0 if convention == "ref" else 1)
    # against the input's size: taps of |sum| 1 in absolute value keep |out| <= max |in|, and a few hundred FP64
    # roundings of values that large stay far below 1e-13
    assert np.abs(got - ref).max() <= 1e-13 * np.abs(x).max(), (convention, radius, fuse, info)


@pytest.mark.parametrize("shape,steps", [("Heat-2D", 82), ("Star2D9P", 5), ("Star2D9P", 125), ("Box2D9P", 64), ("Box2D25P", 125)])
def test_2d_fp64_tile32_gain(ffs, torch_cuda, shape, steps):
    # The mean of the grid is multiplied by (sum w)^T.  Roundings of single outputs average out over 207,000 points; what is left
    # is the gain error that every block shares, from the rounding of the transform matrices and the filter: below half an ulp a
    # block.
    torch = torch_cuda
    _, r, w, _ = ffs.named_stencil(shape, seed=3)
    x = torch.rand((450, 460), dtype=torch.float64, device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    y = torch.empty_like(x)
    with ffs.Plan(2, x.shape, w, r, steps, tile=32) as plan:
        plan.run(x, y)
        torch.cuda.synchronize()
        launches = plan.info["launches"]
    want = x.cpu().numpy().astype(np.longdouble).mean() * np.asarray(w, dtype=np.longdouble).sum() ** steps
    got = y.cpu().numpy().astype(np.longdouble).mean()
    assert abs(got / want - 1) <= 2 ** -53 * launches, (float(got / want - 1), launches)
