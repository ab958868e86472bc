"""The work a user of flashfftstencil_amd has it do, as measurable cases over the ranges it is used in.

A case is a dict: `entry` (plan: Plan.run on device tensors; static: the allocation-free run_static;
batch: Batch.run over independent grids), the stencil by name, the grid, the steps T, the precision form,
the algorithm and the index convention.  One pass is one call: T steps over the whole grid.
"""
import math
import random

import numpy as np
import torch

import flashfftstencil_amd as ffs

SHAPES = {1: ("Heat-1D", "1D5P", "1D7P"), 2: ("Heat-2D", "Box2D9P", "Star2D9P", "Box2D25P"), 3: ("Heat-3D", "Box3D27P")}
RADIUS = {"Heat-1D": 1, "1D5P": 2, "1D7P": 3, "Heat-2D": 1, "Box2D9P": 1, "Star2D9P": 2, "Box2D25P": 2, "Heat-3D": 1,
          "Box3D27P": 1}
TAPS = {"Heat-1D": 3, "1D5P": 5, "1D7P": 7, "Heat-2D": 5, "Box2D9P": 9, "Star2D9P": 9, "Box2D25P": 25, "Heat-3D": 7,
        "Box3D27P": 27}
FORMS = {1: ("fp64", "bf16", "f32"), 2: ("fp64", "f16", "bf16", "f32"), 3: ("fp64", "bf16", "f32")}


def _case(name, entry, shape, n, steps, form="fp64", algorithm="fft", convention="ref", **more):
    n = tuple(n) + (1,) * (3 - len(n))
    c = dict(entry=entry, shape=shape, n0=n[0], n1=n[1], n2=n[2], steps=steps, form=form, algorithm=algorithm,
             convention=convention, **more)
    return dict(c, name=name) if name else c


def listed():
    return [
        # a small grid inside a host loop: a few microseconds of launches
        _case("tiny_box2d9p_fp64", "plan", "Box2D9P", (128, 128), 16),
        # a call inside a captured or allocation-free region: tables and steps in one call
        _case("static_box2d25p_f16", "static", "Box2D25P", (512, 384), 24, "f16"),
        # an image-sized grid with odd sides, T not a multiple of the fused depth
        _case("ragged_star2d9p_f16", "plan", "Star2D9P", (1537, 2003), 50, "f16", convention="centred"),
        # the benchmark's headline: Box2D25P 8192^2 x 256, the fastest form within 1e-6
        _case("box2d25p_8192_f16", "plan", "Box2D25P", (8192, 8192), 256, "f16"),
        # the wide-range mixed form on the same grid
        _case("box2d25p_8192_bf16", "plan", "Box2D25P", (8192, 8192), 64, "bf16"),
        # the FP64 drop-in form: the benchmark's Box2D9P 8192^2 x 128
        _case("box2d9p_8192_fp64", "plan", "Box2D9P", (8192, 8192), 128),
        # the algorithm left to the library, odd sides
        _case("ragged_box2d25p_auto", "plan", "Box2D25P", (2999, 4111), 37, algorithm="auto"),
        # the benchmark's 1D workload: one launch
        _case("heat1d_1m_fp64", "plan", "Heat-1D", (1 << 20,), 64),
        # a long 1D line in the mixed form
        _case("line1d7p_16m_bf16", "plan", "1D7P", ((1 << 24) + 1,), 100, "bf16"),
        # the benchmark's 3D workload
        _case("box3d27p_512_bf16", "plan", "Box3D27P", (512, 512, 512), 32, "bf16"),
        # a 3D grid of odd sides in the drop-in form
        _case("ragged_heat3d_fp64", "plan", "Heat-3D", (201, 187, 230), 20),
        # independent grids advanced together
        _case("batch16_f16", "batch", "", (), 0, "f16", grids=16, grid_seed=4, low=512, high=2048),
    ]


def _spread(rng, lo, hi):
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return v if rng.random() < 0.5 else v | 1


def draw(rng):
    if rng.random() < 0.12:
        return _case(None, "batch", "", (), 0, rng.choice(("fp64", "f16", "bf16")), grids=rng.randint(4, 24),
                     grid_seed=rng.randrange(1 << 20), low=rng.choice((128, 256, 512)), high=rng.choice((1024, 1536, 2048)))
    dims = rng.choice((1, 2, 2, 2, 3))
    shape = rng.choice(SHAPES[dims])
    n = {1: lambda: (_spread(rng, 1 << 12, 1 << 24),),
         2: lambda: (_spread(rng, 96, 8192), _spread(rng, 96, 8192)),
         3: lambda: (_spread(rng, 24, 400), _spread(rng, 24, 400), _spread(rng, 24, 400))}[dims]()
    algorithm = rng.choice(("fft", "fft", "fft", "auto"))
    form = "fp64" if algorithm == "auto" else rng.choice(FORMS[dims])
    points = math.prod(n)
    most = max(4, min({1: 256, 2: 256, 3: 32}[dims], int(2.4e9 / points)))
    steps = _spread(rng, 4, most) if most > 4 else 4
    entry = "static" if points < 4_000_000 and rng.random() < 0.15 else "plan"
    return _case(None, entry, shape, n, steps, form, algorithm, rng.choice(("ref", "centred")))


def _sizes(case):
    return tuple(case["n%d" % d] for d in range(_dims(case)))


def _dims(case):
    return next(d for d in (1, 2, 3) if case["shape"] in SHAPES[d])


def _grids(case):
    """(shape, sizes, steps) of every grid of a batch."""
    rng = random.Random(case["grid_seed"])
    return [(rng.choice(SHAPES[2]), (_spread(rng, case["low"], case["high"]), _spread(rng, case["low"], case["high"])),
             rng.randint(16, 96)) for _ in range(case["grids"])]


def _field(sizes, seed):
    """The grid's values: uniform [0, 1) in 1D and 2D; in 3D eight sinusoids of random phase, amplitude and
    wavevector (up to n/32 periods per axis) plus 1e-3 noise."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    x = torch.rand(sizes, dtype=torch.float64, device="cuda", generator=g)
    if len(sizes) < 3:
        return x
    x *= 1e-3
    rng = random.Random(seed)
    for _ in range(8):
        amp, ph = rng.random() / 8, 2 * math.pi * rng.random()
        arg = torch.full((1, 1, 1), ph, dtype=torch.float64, device="cuda")
        for d, n in enumerate(sizes):
            view = [1, 1, 1]
            view[d] = n
            k = rng.randint(1, max(1, n // 32))
            arg = arg + (2 * math.pi * k / n) * torch.arange(n, dtype=torch.float64, device="cuda").view(view)
        x += amp * torch.cos(arg)
    return x


def _weights(shape):
    return ffs.named_stencil(shape, seed=0x5EED0002)


def prepare(case, seed):
    if case["entry"] == "batch":
        specs, ins = [], []
        for i, (shape, sizes, steps) in enumerate(_grids(case)):
            _, r, w, _ = _weights(shape)
            specs.append(dict(sizes=sizes, weights=w, radius=r, steps=steps))
            ins.append(_field(sizes, seed * 1000 + i))
        return dict(entry="batch", batch=ffs.Batch(specs, precision=case["form"]), ins=ins,
                    outs=[torch.empty_like(x) for x in ins])
    dims, r, w, _ = _weights(case["shape"])
    sizes = _sizes(case)
    x = _field(sizes, seed)
    state = dict(entry=case["entry"], x=x, y=torch.empty_like(x))
    options = dict(precision=case["form"], algorithm=case["algorithm"], convention=case["convention"])
    if case["entry"] == "static":
        state["args"] = (dims, sizes, w, r, case["steps"])
        state["options"] = options
    else:
        state["plan"] = ffs.Plan(dims, sizes, w, r, case["steps"], **options)
    return state


def run(state):
    if state["entry"] == "batch":
        state["batch"].run(state["ins"], state["outs"])
        return state["outs"]
    if state["entry"] == "static":
        ffs.run_static(*state["args"], state["x"], state["y"], **state["options"])
    else:
        state["plan"].run(state["x"], state["y"])
    return state["y"]


def work(case):
    """Each grid read once and written once; one FMA per tap, point and step is what the result needs if
    every step is taken by itself."""
    grids = _grids(case) if case["entry"] == "batch" else [(case["shape"], _sizes(case), case["steps"])]
    return {"bytes": sum(16.0 * math.prod(s) for _, s, _ in grids),
            "flops": sum(2.0 * TAPS[sh] * math.prod(s) * t for sh, s, t in grids)}


def tolerance(case):
    """About four times what the forms show against 64 bits.  FP64: rounding of a few hundred steps.  Mixed
    forms: FP32 sums of split operands (FP32 products in the f32 form), block after block; the 3D field has
    zero mean, so its errors are larger against its own size."""
    if case["form"] == "fp64":
        return {"rel": 2e-13, "max": 2e-12}
    if case["shape"] in SHAPES[3]:
        return {"rel": 1e-6, "max": 1e-5}
    return {"rel": 4e-7, "max": 4e-6} if case["form"] == "f32" else {"rel": 2e-7, "max": 2e-6}


def _exact(shape, sizes, steps, convention, x):
    """T steps as one periodic convolution in FP64: the field's FFT times the T-th power of the taps' FFT."""
    dims, r, w, _ = _weights(shape)
    k = 2 * r + 1
    taps = np.asarray(w).reshape((k,) * dims)
    ker = np.zeros((k,) * dims)
    if convention == "ref":  # out[p] = sum_a w[a] in[p - a]
        ker, first = taps, 0
    else:  # out[p] = sum_o w[o + r] in[p + o]: offset -o for tap o + r
        ker, first = np.flip(taps).copy(), -r
    full = torch.zeros(sizes, dtype=torch.float64, device=x.device)
    at = [torch.from_numpy((np.arange(k) + first) % n).to(x.device) for n in sizes]
    full.index_put_(torch.meshgrid(*at, indexing="ij"), torch.from_numpy(np.ascontiguousarray(ker)).to(x.device),
                    accumulate=True)
    spec = torch.fft.rfftn(full)
    power = torch.polar(spec.abs() ** steps, spec.angle() * steps)
    return torch.fft.irfftn(torch.fft.rfftn(x) * power, s=sizes)


def exact(case, seed):
    if case["entry"] == "batch":
        return [_exact(shape, sizes, steps, "ref", _field(sizes, seed * 1000 + i))
                for i, (shape, sizes, steps) in enumerate(_grids(case))]
    return _exact(case["shape"], _sizes(case), case["steps"], case["convention"], _field(_sizes(case), seed))
