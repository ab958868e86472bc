"""GPU parity of the FP64 form against the FP64 direct-sweep oracle, through the C ABI.

Bar: max|gpu - oracle| / max|oracle| <= 1e-12 for the FP64 form (the stated drop-in tolerance).
Cases follow the reference's shapes and its boundary convention (periodic, ref index convention),
plus the cases the reference cannot run: sizes not divisible by the valid width, grids smaller than a
tile, odd tile counts, T not a multiple of the fused depth, T = 0.
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


SHAPES_2D = ["Heat-2D", "Box2D9P", "Star2D9P", "Box2D25P"]


@pytest.mark.parametrize("shape", SHAPES_2D)
@pytest.mark.parametrize("size", [(37, 53), (16, 16), (5, 7), (64, 40), (1, 19)])
@pytest.mark.parametrize("steps", [1, 2, 5])
def test_2d_fp64_named(ffs, oracle, torch_cuda, shape, size, steps):
    dims, r, w, _ = ffs.named_stencil(shape, seed=7)
    x = oracle.uniform(1234 + size[0] * 31 + size[1], size)
    got, info = _run(ffs, torch_cuda, x, r, w, steps)
    ref = oracle.sweep(x, r, w, steps)
    _, rel, _ = oracle.errors(got, ref)
    print(shape, size, steps, info["fuse"], info["fuse_tail"], rel)
    assert rel <= TOL_FP64, (shape, size, steps, info, rel)


@pytest.mark.parametrize("convention", ["ref", "centred"])
@pytest.mark.parametrize("fuse", [1, 2, 3])
def test_2d_fp64_fuse_and_convention(ffs, oracle, torch_cuda, convention, fuse):
    rng = np.random.default_rng(fuse)
    w = rng.random(9)
    w /= w.sum()
    x = oracle.uniform(99, (45, 61))
    conv = 0 if convention == "ref" else 1
    for steps in (fuse, 2 * fuse + 1, 7):
        got, info = _run(ffs, torch_cuda, x, 1, w, steps, convention=convention, fuse=fuse)
        ref = oracle.sweep(x, 1, w, steps, convention=conv)
        _, rel, _ = oracle.errors(got, ref)
        assert rel <= TOL_FP64, (convention, fuse, steps, info, rel)


def test_2d_unnormalised_weights(ffs, oracle, torch_cuda):
    # weights that neither sum to 1 nor are positive: the spectrum power must still be exact
    rng = np.random.default_rng(3)
    w = rng.standard_normal(25) * 0.3
    x = oracle.uniform(5, (50, 50))
    got, _ = _run(ffs, torch_cuda, x, 2, w, 3)
    ref = oracle.sweep(x, 2, w, 3)
    _, rel, _ = oracle.errors(got, ref)
    assert rel <= TOL_FP64


@pytest.mark.parametrize("shape", ["Heat-1D", "1D5P", "1D7P"])
@pytest.mark.parametrize("n", [1, 7, 240, 241, 1000, 4099])
@pytest.mark.parametrize("steps", [1, 13, 64])
def test_1d_fp64_named(ffs, oracle, torch_cuda, shape, n, steps):
    dims, r, w, _ = ffs.named_stencil(shape, seed=11)
    x = oracle.uniform(777 + n, (n,))
    got, info = _run(ffs, torch_cuda, x, r, w, steps)
    ref = oracle.sweep(x, r, w, steps)
    _, rel, _ = oracle.errors(got, ref)
    assert rel <= TOL_FP64, (shape, n, steps, info, rel)


def test_1d_centred_and_forced_fuse(ffs, oracle, torch_cuda):
    rng = np.random.default_rng(8)
    w = rng.random(5)
    x = oracle.uniform(17, (3001,))
    for fuse in (1, 7, 50):
        for conv in (0, 1):
            got, info = _run(ffs, torch_cuda, x, 2, w / w.sum(), 101, convention=conv, fuse=fuse)
            ref = oracle.sweep(x, 2, w / w.sum(), 101, convention=conv)
            _, rel, _ = oracle.errors(got, ref)
            assert rel <= TOL_FP64, (fuse, conv, info, rel)


def test_zero_steps_is_copy(ffs, oracle, torch_cuda):
    _, r, w, _ = ffs.named_stencil("Box2D9P")
    x = oracle.uniform(1, (33, 17))
    got, _ = _run(ffs, torch_cuda, x, r, w, 0)
    assert np.array_equal(got, x)


def test_deterministic_and_graph_equals_plain(ffs, oracle, torch_cuda):
    torch = torch_cuda
    _, r, w, _ = ffs.named_stencil("Box2D25P", seed=3)
    x = oracle.uniform(2, (200, 150))
    d_in = torch.from_numpy(x).cuda()
    outs = []
    for use_graph in (True, True, False):
        plan = ffs.Plan(2, x.shape, w, r, 9, use_graph=use_graph)
        d_out = torch.empty_like(d_in)
        plan.run(d_in, d_out)
        plan.run(d_in, d_out)  # replay
        torch.cuda.synchronize()
        outs.append(d_out.cpu().numpy())
        plan.close()
    assert np.array_equal(outs[0], outs[1])
    assert np.array_equal(outs[0], outs[2])


def test_run_host_matches_device(ffs, oracle, torch_cuda):
    _, r, w, _ = ffs.named_stencil("Heat-2D", seed=1)
    x = oracle.uniform(3, (70, 30))
    plan = ffs.Plan(2, x.shape, w, r, 6)
    got = plan.run_host(x)
    plan.close()
    ref = oracle.sweep(x, r, w, 6)
    assert oracle.errors(got, ref)[1] <= TOL_FP64


@pytest.mark.parametrize("shape", ["Heat-3D", "Box3D27P"])
@pytest.mark.parametrize("size", [(16, 16, 16), (11, 13, 17), (20, 9, 33), (5, 5, 5), (40, 24, 30)])
@pytest.mark.parametrize("steps", [1, 2, 5])
def test_3d_fp64_named(ffs, oracle, torch_cuda, shape, size, steps):
    _, r, w, _ = ffs.named_stencil(shape, seed=13)
    x = oracle.uniform(3000 + sum(size), size)
    got, info = _run(ffs, torch_cuda, x, r, w, steps)
    ref = oracle.sweep(x, r, w, steps)
    _, rel, _ = oracle.errors(got, ref)
    assert rel <= TOL_FP64, (shape, size, steps, info, rel)


@pytest.mark.parametrize("convention", ["ref", "centred"])
@pytest.mark.parametrize("fuse", [1, 3])
def test_3d_fp64_fuse_convention(ffs, oracle, torch_cuda, convention, fuse):
    rng = np.random.default_rng(70 + fuse)
    w = rng.random(27)
    w /= w.sum()
    x = oracle.uniform(71, (18, 22, 26))
    got, info = _run(ffs, torch_cuda, x, 1, w, 2 * fuse + 1, convention=convention, fuse=fuse)
    ref = oracle.sweep(x, 1, w, 2 * fuse + 1, convention=0 if convention == "ref" else 1)
    assert oracle.errors(got, ref)[1] <= TOL_FP64, info


@pytest.mark.parametrize("precision", ["fp64", "f16", "bf16"])
def test_linear_mapping_is_bitwise_equal(ffs, oracle, torch_cuda, precision):
    # the wave-to-tile mapping only reorders independent tile pairs: results are bitwise identical
    torch = torch_cuda
    _, r, w, _ = ffs.named_stencil("Box2D25P", seed=8)
    x = oracle.uniform(31, (333, 290))
    d_in = torch.from_numpy(x).cuda()
    outs = []
    for mapping in ("xcd", "linear"):
        plan = ffs.Plan(2, x.shape, w, r, 11, precision=precision, mapping=mapping)
        assert plan.info["mapping"] == (1 if mapping == "xcd" else 2)
        d_out = torch.empty_like(d_in)
        plan.run(d_in, d_out)
        torch.cuda.synchronize()
        outs.append(d_out.cpu().numpy())
        plan.close()
    assert np.array_equal(outs[0], outs[1])


@pytest.mark.parametrize("algorithm,precision", [("fft", "fp64"), ("fft", "f16"), ("direct", "fp64")])
def test_run_captured_in_caller_graph(ffs, oracle, torch_cuda, algorithm, precision):
    # with use_graph = 0 a run only enqueues kernels on the caller's stream, so it can be recorded into the
    # caller's own graph; every replay (with eager work in between) must equal the eager result
    torch = torch_cuda
    _, r, w, _ = ffs.named_stencil("Box2D25P", seed=12)
    x = oracle.uniform(41, (200, 180))
    d_in = torch.from_numpy(x).cuda()
    plan = ffs.Plan(2, x.shape, w, r, 9, precision=precision, algorithm=algorithm, use_graph=False)
    eager = torch.empty_like(d_in)
    plan.run(d_in, eager)
    torch.cuda.synchronize()
    out = torch.empty_like(d_in)
    g = torch.cuda.CUDAGraph()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        plan.run(d_in, out)  # warm-up on the side stream before capture
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    with torch.cuda.graph(g):
        plan.run(d_in, out)
    for k in range(3):
        out.zero_()
        scratch = torch.ones(1000, device="cuda") * k  # eager work between replays
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager), (k, float(scratch.sum()))
    plan.close()


def test_fill_uniform_device_matches_host(ffs, oracle, torch_cuda):
    torch = torch_cuda
    d = torch.empty(100003, dtype=torch.float64, device="cuda")
    ffs.fill_uniform_device(0x5EED0002, d)
    torch.cuda.synchronize()
    assert np.array_equal(d.cpu().numpy(), ffs.fill_uniform(0x5EED0002, d.numel()))


def test_planner_heat1d_single_launch(ffs, torch_cuda):
    # 2^20 points x 64 steps: the run is launch-bound, and the planner's whole-run model takes the one
    # block of depth 64 (V = 112 of the 240-point window) over two blocks of depth 32.
    _, r, w, _ = ffs.named_stencil("Heat-1D", seed=1)
    plan = ffs.Plan(1, (1 << 20,), w, r, 64, precision="fp64")
    info = plan.info
    plan.close()
    assert info["fuse"] == 64 and info["blocks"] == 1 and info["valid"][0] == 112, info


@pytest.mark.parametrize("precision", ["fp64", "f16"])
def test_graph_cache_cycles_buffer_pairs(ffs, oracle, torch_cuda, precision):
    # one plan driven with five (d_in, d_out) pairs in turn, twice round: the plan keeps the captured chains
    # of four pairs, so the fifth evicts the least recently used one and every pair is re-captured on its
    # next turn; every run must equal the first run of its input bitwise, and the FP64 ones the oracle
    torch = torch_cuda
    _, r, w, _ = ffs.named_stencil("Box2D9P", seed=13)
    plan = ffs.Plan(2, (96, 80), w, r, 48, precision=precision, fuse=4)
    assert plan.info["blocks"] > 4  # graph replay is used
    xs = [oracle.uniform(60 + i, (96, 80)) for i in range(5)]
    ins = [torch.from_numpy(x).cuda() for x in xs]
    outs = [torch.empty_like(d) for d in ins]
    first = []
    for rnd in range(2):
        for i in range(5):
            outs[i].fill_(float("nan"))
            plan.run(ins[i], outs[i])
            torch.cuda.synchronize()
            if rnd == 0:
                first.append(outs[i].clone())
            else:
                assert torch.equal(outs[i], first[i]), i
    tol = 1e-12 if precision == "fp64" else 1e-6
    for i in range(5):
        assert oracle.errors(first[i].cpu().numpy(), oracle.sweep(xs[i], r, w, 48))[1] <= tol
    plan.close()


@pytest.mark.parametrize("radius", [2, 3])
@pytest.mark.parametrize("precision,algorithm", [("fp64", "fft"), ("bf16", "fft"), ("f32", "fft"), ("fp64", "auto")])
@pytest.mark.parametrize("convention", ["ref", "centred"])
def test_3d_wider_stencils(ffs, oracle, torch_cuda, radius, precision, algorithm, convention):
    """Custom 3D stencils wider than the named ones (5^3 and 7^3 random weights): the 16^3 tiles then
    keep V = 16 - 2 r t (down to 4), with tails; ragged grids; against the oracle at the form's bar.
    AUTO takes the FFT path here (the direct kernels stop at radius 1 in 3D)."""
    rng = np.random.default_rng(40 + radius)
    w = rng.random((2 * radius + 1) ** 3)
    w /= w.sum()
    tol = 1e-12 if precision == "fp64" else 1e-6
    for sizes, steps in [((23, 19, 29), 1), ((17, 26, 21), 3), ((30, 14, 33), 5)]:
        x = oracle.uniform(7 * radius + steps, sizes)
        try:
            plan = ffs.Plan(3, sizes, w, radius, steps, precision=precision, algorithm=algorithm,
                            convention=convention)
        except ffs.FFSError as e:
            pytest.fail(f"plan rejected: radius {radius} {precision} {algorithm}: {e}")
        d_in = torch_cuda.from_numpy(x).cuda()
        d_out = torch_cuda.empty_like(d_in)
        plan.run(d_in, d_out)
        torch_cuda.cuda.synchronize()
        info = plan.info
        plan.close()
        ref = oracle.sweep(x, radius, w, steps, convention=0 if convention == "ref" else 1)
        rel = oracle.errors(d_out.cpu().numpy(), ref)[1]
        assert rel <= tol, (radius, precision, algorithm, convention, sizes, steps, info, rel)


@pytest.mark.parametrize("radius", [2, 3])
def test_3d_direct_refuses_wider_stencils(ffs, torch_cuda, radius):
    """The direct kernels cover radius <= 1 in 3D; wider stencils are a clear FFS_ERR_UNSUPPORTED."""
    w = np.full((2 * radius + 1) ** 3, 1.0 / (2 * radius + 1) ** 3)
    with pytest.raises(ffs.FFSError, match="not offered in 3D"):
        ffs.Plan(3, (20, 20, 20), w, radius, 2, precision="fp64", algorithm="direct")


@pytest.mark.parametrize("dims,radius", [(2, 5), (2, 7), (1, 5), (1, 12)])
@pytest.mark.parametrize("weights", ["signed", "growing"])
def test_wide_stencils_unusual_weights(ffs, oracle, torch_cuda, dims, radius, weights):
    """Wide custom stencils in 1D and 2D, every FFT form the dimension offers, with weights that are not
    a positive normalised set: signed taps summing to 1 (an oscillating kernel) or positive taps summing
    to 1.3 (a growing field, so the DC gain (sum w)^t and the mixed forms' tile scales are exercised)."""
    rng = np.random.default_rng(10 * dims + radius)
    n = (2 * radius + 1) ** dims
    if weights == "signed":
        w = rng.random(n) - 0.45
        w /= w.sum()
    else:
        w = rng.random(n)
        w *= 1.3 / w.sum()
    sizes = (3001,) if dims == 1 else (71, 90)
    steps = 6
    x = oracle.uniform(31 * radius, sizes)
    ref = oracle.sweep(x, radius, w, steps)
    forms = ["fp64", "bf16", "f32"] + (["f16"] if dims == 2 else [])
    for form in forms:
        plan = ffs.Plan(dims, sizes, w, radius, steps, precision=form)
        d_in = torch_cuda.from_numpy(x).cuda()
        d_out = torch_cuda.empty_like(d_in)
        plan.run(d_in, d_out)
        torch_cuda.cuda.synchronize()
        info = plan.info
        plan.close()
        rel = oracle.errors(d_out.cpu().numpy(), ref)[1]
        assert rel <= (1e-12 if form == "fp64" else 1e-6), (dims, radius, weights, form, info, rel)


@pytest.mark.parametrize("precision", ["fp64", "bf16"])
def test_3d_mappings_bitwise_equal(ffs, oracle, torch_cuda, precision):
    """The 3D kernel's wave-to-tile orders (XCD bands: the mixed form's default; hardware order: the FP64
    form's) only reorder independent tile pairs: bitwise equal results, both against the oracle."""
    _, r, w, _ = ffs.named_stencil("Box3D27P", seed=5)
    x = oracle.uniform(77, (40, 24, 30))
    outs = []
    for mapping in ("xcd", "linear", "auto"):
        plan = ffs.Plan(3, x.shape, w, r, 5, precision=precision, mapping=mapping)
        info = plan.info
        d_in = torch_cuda.from_numpy(x).cuda()
        d_out = torch_cuda.empty_like(d_in)
        plan.run(d_in, d_out)
        torch_cuda.cuda.synchronize()
        plan.close()
        outs.append(d_out.cpu().numpy())
        if mapping == "auto":
            assert info["mapping"] == (2 if precision == "fp64" else 1), info
    assert np.array_equal(outs[0], outs[1]) and np.array_equal(outs[0], outs[2])
    assert oracle.errors(outs[0], oracle.sweep(x, r, w, 5))[1] <= (1e-12 if precision == "fp64" else 1e-6)


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("bf16", 1e-6)])
@pytest.mark.parametrize("convention", ["ref", "centred"])
@pytest.mark.parametrize("radius,sizes,steps", [(1, (150, 131, 139), 7), (1, (127, 130, 141), 12), (1, (3, 400, 380), 5),
                                                (1, (260, 78, 84), 2), (2, (121, 113, 140), 3), (3, (90, 131, 157), 2),
                                                (1, (129, 257, 65), 1)])
def test_3d_streamed(ffs, oracle, torch_cuda, precision, tol, convention, radius, sizes, steps):
    """3D grids around the size from which the streamed kernel is the faster one (which kernel runs is the planner's choice
    here; test_3d_streamed_forms asserts it): planes one past and one short of a multiple of the valid width, segments of
    unequal length, few planes, signed taps."""
    torch = torch_cuda
    rng = np.random.default_rng(40 * radius + steps)
    w = rng.standard_normal((2 * radius + 1) ** 3)
    w += 2.0 * np.abs(w).sum() / w.size
    w /= w.sum()
    x = oracle.uniform(300 + steps, sizes)
    d_in = torch.from_numpy(x).cuda()
    d_out = torch.empty_like(d_in)
    with ffs.Plan(3, sizes, w, radius, steps, precision=precision, convention=convention) as plan:
        plan.run(d_in, d_out)
        torch.cuda.synchronize()
        info = plan.info
    ref = oracle.sweep(x, radius, w, steps, convention=0 if convention == "ref" else 1)
    rel = oracle.errors(d_out.cpu().numpy(), ref)[1]
    assert rel <= tol, (precision, convention, radius, sizes, steps, info, rel)


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("bf16", 1e-6)])
@pytest.mark.parametrize("convention", ["ref", "centred"])
@pytest.mark.parametrize("radius,n,steps", [(1, 256, 7), (1, 257, 8), (1, 255, 9), (1, 1023, 64), (3, 10, 50), (1, 1, 3),
                                            (2, 4099, 130), (1, 5000, 248), (12, 1500, 30), (40, 700, 2), (60, 2000, 9)])
def test_1d_banded_product(ffs, oracle, torch_cuda, precision, tol, convention, radius, n, steps):
    """1D runs as banded products: grids around a tile of 256 outputs, smaller than the stencil's reach, numbers of
    taps around a multiple of the contraction block (2rt + 16 = 16 b, 32 b and one past), up to the deepest launch and past it,
    wide stencils, signed taps."""
    torch = torch_cuda
    rng = np.random.default_rng(radius + steps)
    w = rng.standard_normal(2 * radius + 1)
    w += 2.0 * np.abs(w).sum() / w.size
    w /= w.sum()
    x = oracle.uniform(70 + n, (n,))
    d_in = torch.from_numpy(x).cuda()
    d_out = torch.empty_like(d_in)
    with ffs.Plan(1, (n,), w, radius, steps, precision=precision, convention=convention) as plan:
        plan.run(d_in, d_out)
        torch.cuda.synchronize()
        info = plan.info
    ref = oracle.sweep(x, radius, w, steps, convention=0 if convention == "ref" else 1)
    rel = oracle.errors(d_out.cpu().numpy(), ref)[1]
    assert rel <= tol, (precision, convention, radius, n, steps, info, rel)


@pytest.mark.parametrize("n", [(1 << 22) + 8191, (1 << 21) + 13])
def test_1d_banded_product_large(ffs, torch_cuda, n):
    """Several windows per wave, the next one requested ahead: the two-tile variant of the mixed kernel (above 4 Mi points)
    and the one-tile variant, against the FP64 form, ragged lengths."""
    torch = torch_cuda
    _, r, w, _ = ffs.named_stencil("1D7P", seed=2)
    d_in = torch.empty(n, dtype=torch.float64, device="cuda")
    ffs.fill_uniform_device(3, d_in)
    outs = []
    for precision in ("bf16", "fp64"):
        with ffs.Plan(1, tuple(d_in.shape), w, r, 71, precision=precision) as plan:
            d = torch.empty_like(d_in)
            plan.run(d_in, d)
            torch.cuda.synchronize()
        outs.append(d)
    assert float((outs[0] - outs[1]).abs().max() / outs[1].abs().max()) <= 1e-6


@pytest.mark.parametrize("convention", ["ref", "centred"])
@pytest.mark.parametrize("shape,sizes,steps", [("Box3D27P", (150, 128, 201), 8), ("Heat-3D", (131, 170, 140), 20)])
@pytest.mark.parametrize("field", ["waves", "ramp", "bumps"])
def test_3d_streamed_smooth_fields_as_exact_as_blocks(ffs, oracle, torch_cuda, convention, shape, sizes, steps, field):
    """Fields that vary over one to several planes' windows: the streamed BF16 runs (planes relative to a fitted plane) are no
    less exact than the 16^3 blocks they stand for, run one by one (0.39 to 0.66 of their error here, with a mean in place of
    the plane up to 1.49)."""
    torch = torch_cuda
    _, r, w, _ = ffs.named_stencil(shape, seed=0x5EED0002)
    g = np.meshgrid(*[np.arange(n) / n for n in sizes], indexing="ij")
    if field == "waves":
        x = 0.3 * np.cos(2 * np.pi * (g[0] + g[1] + 0.1)) + 0.2 * np.cos(2 * np.pi * (g[1] - 2 * g[2])) + 0.2 * np.sin(
            2 * np.pi * (2 * g[0] + g[2]))
    elif field == "ramp":
        x = 3.0 * g[0] + g[1] - 2.0 * g[2]
    else:
        x = sum(np.exp(-sum(((a - b) * n) ** 2 for a, b, n in zip(g, at, sizes)) / s ** 2)
                for at, s in (((0.3, 0.4, 0.6), 30), ((0.7, 0.6, 0.3), 25), ((0.5, 0.8, 0.8), 40)))
    x = np.ascontiguousarray(x)
    ref = oracle.sweep(x, r, w, steps, convention=0 if convention == "ref" else 1)
    d_in = torch.from_numpy(x).cuda()
    d_out = torch.empty_like(d_in)
    with ffs.Plan(3, sizes, w, r, steps, precision="bf16", convention=convention) as plan:
        plan.run(d_in, d_out)
        a, b = d_in.clone(), torch.empty_like(d_in)
        info = plan.info
        for k in range(info["blocks"]):
            plan.run_block(a, b, tail=k == info["blocks"] - 1)
            a, b = b, a
        torch.cuda.synchronize()
    run = oracle.errors(d_out.cpu().numpy(), ref)[2]
    blocks = oracle.errors(a.cpu().numpy(), ref)[2]
    assert run <= blocks, (run, blocks, info)


def _signed_mean_one(radius, dims, seed):
    rng = np.random.default_rng(seed)
    w = rng.standard_normal((2 * radius + 1) ** dims)
    w += 2.0 * np.abs(w).sum() / w.size
    return w / w.sum()


@pytest.mark.parametrize("convention", ["ref", "centred"])
@pytest.mark.parametrize("precision,radius,sizes,steps,depth,launches", [
    ("fp64", 1, (129, 257, 65), 1, 1, 1), ("fp64", 1, (2, 600, 610), 5, 1, 5), ("fp64", 1, (150, 131, 139), 7, 2, 4),
    ("fp64", 1, (2, 900, 800), 4, 2, 2), ("fp64", 2, (121, 113, 140), 3, 1, 3), ("fp64", 2, (3, 700, 690), 2, 1, 2),
    ("bf16", 1, (129, 257, 65), 1, 1, 1), ("bf16", 1, (3, 900, 900), 4, 1, 4), ("bf16", 1, (150, 131, 139), 7, 2, 4),
    ("bf16", 1, (2, 600, 610), 5, 2, 3), ("bf16", 1, (5, 1000, 1000), 11, 3, 4), ("bf16", 2, (140, 150, 160), 3, 1, 3),
    ("bf16", 3, (90, 131, 157), 2, 1, 2), ("bf16", 3, (5, 500, 500), 2, 1, 2)])
def test_3d_streamed_forms(ffs, oracle, torch_cuda, convention, precision, radius, sizes, steps, depth, launches):
    """The streamed kernel in every form: 3, 5 and 7 taps along axis 0 (FP64 3 and 5), a last launch of a smaller depth (padded
    taps), fewer planes than taps, signed taps.  The route and its depth are asserted."""
    torch = torch_cuda
    w = _signed_mean_one(radius, 3, 40 * radius + steps)
    x = oracle.uniform(300 + steps, sizes)
    d_in = torch.from_numpy(x).cuda()
    d_out = torch.empty_like(d_in)
    with ffs.Plan(3, sizes, w, radius, steps, precision=precision, convention=convention) as plan:
        plan.run(d_in, d_out)
        torch.cuda.synchronize()
        info = plan.info
    assert (info["run_kernel"], info["run_depth"], info["launches"]) == (ffs.RUN_KERNELS["stream"], depth, launches), info
    ref = oracle.sweep(x, radius, w, steps, convention=0 if convention == "ref" else 1)
    assert oracle.errors(d_out.cpu().numpy(), ref)[1] <= (1e-12 if precision == "fp64" else 1e-6), info


@pytest.mark.parametrize("convention", ["ref", "centred"])
@pytest.mark.parametrize("precision,radius,n,steps,depth,launches", [
    ("fp64", 3, 900, 101, 51, 2), ("fp64", 60, 2000, 10, 4, 3), ("fp64", 3, 700, 83, 42, 2), ("fp64", 1, 3001, 249, 125, 2),
    ("fp64", 100, 3000, 5, 2, 3), ("bf16", 3, 900, 101, 34, 3), ("bf16", 60, 2000, 9, 2, 5), ("bf16", 2, 500, 249, 63, 4),
    ("bf16", 24, 400, 21, 6, 4)])
def test_1d_banded_product_tails(ffs, oracle, torch_cuda, convention, precision, radius, n, steps, depth, launches):
    """Banded products whose last launch has another depth (its own taps and, in the mixed form, operands), wide and narrow
    stencils; the route and its depth are asserted."""
    torch = torch_cuda
    assert steps % depth != 0 and -(-steps // depth) == launches
    w = _signed_mean_one(radius, 1, radius + steps)
    x = oracle.uniform(70 + n, (n,))
    d_in = torch.from_numpy(x).cuda()
    d_out = torch.empty_like(d_in)
    with ffs.Plan(1, (n,), w, radius, steps, precision=precision, convention=convention) as plan:
        plan.run(d_in, d_out)
        torch.cuda.synchronize()
        info = plan.info
    assert (info["run_kernel"], info["run_depth"], info["launches"]) == (ffs.RUN_KERNELS["line"], depth, launches), info
    ref = oracle.sweep(x, radius, w, steps, convention=0 if convention == "ref" else 1)
    assert oracle.errors(d_out.cpu().numpy(), ref)[1] <= (1e-12 if precision == "fp64" else 1e-6), info


@pytest.mark.parametrize("convention", ["ref", "centred"])
@pytest.mark.parametrize("dims,sizes,radius,fuse,steps,precision,algorithm,kernel", [
    (1, (2000,), 1, 50, 130, "fp64", "fft", "line"), (1, (2000,), 3, 20, 47, "fp64", "fft", "line"),
    (1, (700,), 2, 30, 71, "bf16", "fft", "line"), (1, (241,), 3, 37, 75, "bf16", "fft", "line"),
    (1, (5000,), 1, 40, 100, "fp64", "direct", "line"), (1, (3000,), 2, 17, 40, "fp64", "direct", "line"),
    (1, (2500,), 3, 9, 22, "fp64", "direct", "line"),
    (2, (75, 90), 2, 4, 11, "f16", "fft", "wide"), (2, (75, 90), 2, 4, 11, "bf16", "fft", "wide"),
    (2, (33, 61), 1, 8, 21, "f16", "fft", "wide"), (2, (33, 61), 3, 3, 8, "bf16", "fft", "wide"),
    (2, (64, 48), 1, 15, 40, "f16", "fft", "wide"),
    (3, (150, 131, 139), 1, 2, 7, "fp64", "fft", "stream"), (3, (150, 131, 139), 1, 2, 7, "bf16", "fft", "stream")])
def test_run_block_where_runs_launch_other_kernels(ffs, oracle, torch_cuda, convention, dims, sizes, radius, fuse, steps,
                                                   precision, algorithm, kernel):
    """ffs_run_block, main and tail, on plans whose whole runs launch other kernels: the 240-point windows, k_direct1d, the
    32-point mixed tiles with V <= 16 and the 16^3 tiles."""
    torch = torch_cuda
    w = _signed_mean_one(radius, dims, 9 * radius + fuse)
    x = oracle.uniform(11 + fuse, sizes)
    d_in = torch.from_numpy(x).cuda()
    with ffs.Plan(dims, sizes, w, radius, steps, precision=precision, convention=convention, fuse=fuse,
                  algorithm=algorithm) as plan:
        info = plan.info
        assert info["run_kernel"] == ffs.RUN_KERNELS[kernel] and info["fuse"] == fuse and info["fuse_tail"] == steps % fuse
        for tail in (False, True):
            d_out = torch.empty_like(d_in)
            plan.run_block(d_in, d_out, tail=tail)
            torch.cuda.synchronize()
            ref = oracle.sweep(x, radius, w, info["fuse_tail"] if tail else fuse, convention=0 if convention == "ref" else 1)
            tol = 1e-12 if precision == "fp64" else 1e-6
            assert oracle.errors(d_out.cpu().numpy(), ref)[1] <= tol, (tail, info)


@pytest.mark.parametrize("dims,sizes,radius,precision,algorithm,fuses", [
    (1, (3001,), 1, "fp64", "fft", (1, 7, 50, 100)), (1, (3001,), 2, "bf16", "fft", (1, 9, 50)),
    (1, (3001,), 1, "fp64", "direct", (1, 7, 60)), (1, (3001,), 3, "fp64", "auto", (2, 9)),
    (3, (150, 131, 139), 1, "fp64", "fft", (1, 2)), (3, (150, 131, 139), 1, "bf16", "fft", (1, 2, 3)),
    (3, (150, 131, 139), 1, "fp64", "fft", (4,))])
def test_forced_depth_is_the_launched_depth(ffs, oracle, torch_cuda, dims, sizes, radius, precision, algorithm, fuses):
    """A depth that the caller sets is what 1D and 3D runs launch (4 in 3D: beyond the streamed kernel's, on the tiles)."""
    torch = torch_cuda
    w = _signed_mean_one(radius, dims, radius)
    steps = 101 if dims == 1 else 7
    x = oracle.uniform(5, sizes)
    d_in = torch.from_numpy(x).cuda()
    ref = oracle.sweep(x, radius, w, steps)
    for fuse in fuses:
        d_out = torch.empty_like(d_in)
        with ffs.Plan(dims, sizes, w, radius, steps, precision=precision, algorithm=algorithm, fuse=fuse) as plan:
            plan.run(d_in, d_out)
            torch.cuda.synchronize()
            info = plan.info
        assert info["run_depth"] == fuse and info["launches"] == -(-steps // fuse), (fuse, info)
        assert oracle.errors(d_out.cpu().numpy(), ref)[1] <= (1e-12 if precision == "fp64" else 1e-6), (fuse, info)


@pytest.mark.parametrize("shape,steps", [("Heat-3D", 26), ("Box3D27P", 31)])
def test_3d_streamed_fp64_gain(ffs, torch_cuda, shape, steps):
    """The mean of the grid is multiplied by (sum w)^T.  Roundings of single outputs average out over 3.4 million points; what
    is left is the gain error that every launch shares, from the rounding of the transform matrices and the filters: below half
    an ulp a launch."""
    torch = torch_cuda
    _, r, w, _ = ffs.named_stencil(shape, seed=0x5EED0002)
    x = torch.rand((140, 150, 160), dtype=torch.float64, device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    y = torch.empty_like(x)
    with ffs.Plan(3, x.shape, w, r, steps) as plan:
        plan.run(x, y)
        torch.cuda.synchronize()
        info = plan.info
    assert info["run_kernel"] == ffs.RUN_KERNELS["stream"]
    want = x.cpu().numpy().astype(np.longdouble).mean() * np.asarray(w, dtype=np.longdouble).sum() ** steps
    got = y.cpu().numpy().astype(np.longdouble).mean()
    assert abs(got / want - 1) <= 2 ** -53 * info["launches"], (float(got / want - 1), info)
