"""Unit checks of the plan tables the GPU generates (read back with ffs_plan_read_table), against closed
forms, so that a wrong DFT entry, sign, index map or normalisation is found in the table itself and not
only through an end-to-end result:
  * DFT operands: F[j][k] = exp(-2 pi i j k / L) and F F^H = L I, in every family's per-lane layout
    (reference: src/2D/create_fft_pfa_plan.cu:25-39, src/1D/create_fft_pfa_plan.cu:43-76);
  * split operands of the mixed forms: the terms sum back to F within the split's precision, and the
    FP32 operands with their low-order terms give F to ~2^-48;
  * spectra: H = K^t / prod(P) against a numpy FFT of the zero-padded kernel, K(0)^t = (sum w)^t, and
    the Heat-1D closed form K^t = ((1 + cos th)/2)^t e^{-i th t} on the 240-point prime-factor map
    (reference: src/2D/create_fft_pfa_plan.cu:76-107, src/1D/create_fft_pfa_plan.cu:143-178).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def dft(L):
    """F[j][k] = exp(-2 pi i j k / L) with the angle reduced exactly, (j k mod L) / L, before the
    exponential (numpy's own rounding of 2 pi j k / L for large j k would exceed the tables' error)."""
    j = np.arange(L)
    return np.exp(-2j * np.pi * (np.outer(j, j) % L) / L)


def table(plan, which, dtype):
    return np.frombuffer(plan.read_table(which), dtype=dtype)


def check_dft(F, L):
    assert np.abs(F - dft(L)).max() < 4e-16 * L
    assert np.abs(F @ F.conj().T - L * np.eye(L)).max() < 1e-13


def ops16(plan, axis):
    """16-point operands of one axis: [arr: Fr, -(Fr+Fi), Fi-Fr][chunk c][lane], entry (4c + lane/16, lane%16)."""
    t = table(plan, 0, np.float64)[axis * 768:(axis + 1) * 768].reshape(3, 4, 64)
    R, S, D = (np.zeros((16, 16)) for _ in range(3))
    for c in range(4):
        for lane in range(64):
            row, col = 4 * c + lane // 16, lane % 16
            R[row, col], S[row, col], D[row, col] = t[0, c, lane], t[1, c, lane], t[2, c, lane]
    return R, S, D


def gauss_arrays(arrays, F):
    """The three arrays of the Gauss form, each generated in FP64 from the exact entry: R = Re F,
    S = -(Re F + Im F), D = Im F - Re F, each checked against the closed form F on its own (recovering
    Im F from D + R rounds, so the arrays are not compared with each other bitwise)."""
    R, S, D = arrays
    tol = 4e-16 * F.shape[0]
    assert np.abs(R - F.real).max() < tol
    assert np.abs(S + F.real + F.imag).max() < tol
    assert np.abs(D - (F.imag - F.real)).max() < tol
    return R + 1j * (D + R)


def test_dft_operands_16(ffs, torch_cuda):
    _, r, w, _ = ffs.named_stencil("Box2D9P", seed=1)
    plan = ffs.Plan(2, (64, 64), w, r, 3, precision="fp64", tile=16)
    for axis in (0, 1):
        check_dft(gauss_arrays(ops16(plan, axis), dft(16)), 16)
    plan.close()


def test_dft_operands_1d_prime_factor(ffs, torch_cuda):
    # the 240-point window runs as a 15 x 16 Good-Thomas matrix: axis 0 holds F_15 zero-padded to 16
    plan = ffs.Plan(1, (5000,), np.array([0.25, 0.5, 0.25]), 1, 8, precision="fp64")
    want = np.zeros((16, 16), complex)
    want[:15, :15] = dft(15)
    F15 = gauss_arrays(ops16(plan, 0), want)
    check_dft(F15[:15, :15], 15)
    assert np.all(F15[15, :] == 0) and np.all(F15[:, 15] == 0)
    check_dft(gauss_arrays(ops16(plan, 1), dft(16)), 16)
    plan.close()


def test_dft_operands_32_fp64(ffs, torch_cuda):
    # What ffs_plan_read_table answers for a plan of 32-point FP64 tiles; its kernels read the real half-sample tables
    # (test_real_tables_32_fp64).  [R][chunk v][column block Kb][arr][lane], lane (n + 16k) = entry (16 R + 4 v + k, 16 Kb + n)
    _, r, w, _ = ffs.named_stencil("Box2D25P", seed=2)
    plan = ffs.Plan(2, (256, 256), w, r, 8, precision="fp64", tile=32)
    assert plan.info["tile"][0] == 32
    t = table(plan, 0, np.float64)[:3072].reshape(2, 4, 2, 3, 64)
    R, S, D = (np.zeros((32, 32)) for _ in range(3))
    for Rb in range(2):
        for v in range(4):
            for Kb in range(2):
                for lane in range(64):
                    row, col = 16 * Rb + 4 * v + lane // 16, 16 * Kb + lane % 16
                    R[row, col], S[row, col], D[row, col] = t[Rb, v, Kb, :, lane]
    check_dft(gauss_arrays((R, S, D), dft(32)), 32)
    plan.close()


def _split_terms(words, f16):
    """[arr][Kb][term][word][lane] words of two 16-bit values -> per-term 32 x 32 matrices of arr."""
    w = words.reshape(3, 2, 3, 4, 64)
    half = np.float16 if f16 else None
    out = np.zeros((3, 3, 32, 32))
    for arr in range(3):
        for Kb in range(2):
            for term in range(3):
                for wd in range(4):
                    for lane in range(64):
                        word = int(w[arr, Kb, term, wd, lane])
                        for h in range(2):
                            bits = (word >> (16 * h)) & 0xFFFF
                            if f16:
                                val = float(np.array([bits], dtype=np.uint16).view(half)[0])
                            else:
                                val = float(np.array([bits << 16], dtype=np.uint32).view(np.float32)[0])
                            e = 2 * wd + h
                            row, col = 16 * (e >> 2) + 4 * (lane // 16) + (e & 3), 16 * Kb + lane % 16
                            out[arr, term, row, col] = val
    return out


@pytest.mark.parametrize("form,bound", [("bf16", 2.0 ** -24), ("f16", 2.0 ** -22)])
def test_split_operands_32(ffs, torch_cuda, form, bound):
    # BF16: F = h + m + l (3 terms, ~24 bits); FP16: F = h + l (2 terms, ~22 bits); arrays Fr, Fi, -Fi
    _, r, w, _ = ffs.named_stencil("Box2D25P", seed=3)
    plan = ffs.Plan(2, (256, 256), w, r, 8, precision=form)
    terms = _split_terms(table(plan, 1, np.uint32)[:4608], form == "f16")
    F = dft(32)
    for arr, want in enumerate((F.real, F.imag, -F.imag)):
        got = terms[arr].sum(axis=0)
        assert np.abs(got - want).max() <= bound, (form, arr)
        if form == "f16":
            assert np.all(terms[arr, 2] == 0)  # no third FP16 term
    plan.close()


def test_split_operands_16(ffs, torch_cuda):
    """16-point mixed operands (a 3D plan: every axis 16 points).  BF16 words [axis][arr][pairing][word]
    [lane], element e of lane (j + 16q) = row 4q + (e & 3), column j; pairings 0, 1, 2 carry the terms
    h, m, l in their first four elements, which sum back to F within the 3-term split's precision.  FP32
    chunks [axis][arr][c][lane] = F[4q + c][j] rounded to FP32, then their low-order terms, with which
    they give F to ~2^-48 (the 3D FP32 form's compensated matrix)."""
    with ffs.Plan(3, (32, 32, 32), np.full(27, 1 / 27), 1, 2, precision="f32") as plan:
        words = table(plan, 1, np.uint32)
    F = dft(16)
    wants = (F.real, F.imag, -F.imag)
    bf = words[:3 * 3072].reshape(3, 3, 4, 4, 64)
    f32 = words[3 * 3072:3 * 3072 + 2 * 3 * 768].view(np.float32).astype(np.float64)
    hi, lo = f32[:2304].reshape(3, 3, 4, 64), f32[2304:].reshape(3, 3, 4, 64)
    lanes = np.arange(64)
    rows_c = 4 * (lanes // 16)
    cols = lanes % 16
    for axis in range(3):
        for arr, want in enumerate(wants):
            split = np.zeros((16, 16))
            for g in range(3):
                for wd in range(2):  # elements 0..3: words 0 and 1
                    for h in range(2):
                        bits = ((bf[axis, arr, g, wd] >> (16 * h)) & 0xFFFF).astype(np.uint32) << 16
                        split[rows_c + 2 * wd + h, cols] += bits.view(np.float32).astype(np.float64)
            assert np.abs(split - want).max() <= 2.0 ** -24, (axis, arr)
            H, L = np.zeros((16, 16)), np.zeros((16, 16))
            for c in range(4):
                H[rows_c + c, cols] = hi[axis, arr, c]
                L[rows_c + c, cols] = lo[axis, arr, c]
            assert np.abs(H - want).max() <= 2.0 ** -25, (axis, arr)  # FP32 rounding of entries <= 1
            assert np.abs(H + L - want).max() <= 2.0 ** -46, (axis, arr)
            assert np.abs(H - want).max() > 2.0 ** -30  # the low-order terms carry something


def spectrum(plan, length):
    t = table(plan, 2, np.float64)
    main = t[:length] + 1j * t[length:2 * length]
    tail = t[2 * length:3 * length] + 1j * t[3 * length:4 * length]
    return main, tail


def kernel_dft(w, radius, dims, P, convention):
    K = 2 * radius + 1
    ker = np.zeros((P,) * dims)
    ker[(slice(0, K),) * dims] = np.asarray(w).reshape((K,) * dims)
    if convention == "centred":  # out[p] = sum_o w[o + r] in[p + o]: taps at offsets r - a
        ker = np.zeros((P,) * dims)
        for a in np.ndindex(*(K,) * dims):
            ker[tuple((radius - ai) % P for ai in a)] += np.asarray(w).reshape((K,) * dims)[a]
    return np.fft.fftn(ker)


@pytest.mark.parametrize("convention", ["ref", "centred"])
@pytest.mark.parametrize("form", ["fp64", "f16"])
def test_spectrum_2d32(ffs, torch_cuda, convention, form):
    # entry e = (kb * 4 + v) * 64 + lane of block kb = 2 Rb + C: row 16 Rb + (q + 4 v | 4 q + v), column
    # 16 C + j (FP64 | FP32 accumulator order); unnormalised weights (sum 1.3), main depth 4 and tail 1
    rng = np.random.default_rng(5)
    w = rng.random(25)
    w *= 1.3 / w.sum()
    plan = ffs.Plan(2, (200, 200), w, 2, 9, precision=form, convention=convention, fuse=4, tile=32)
    info = plan.info
    assert (info["fuse"], info["fuse_tail"]) == (4, 1)
    main, tail = spectrum(plan, 1024)
    Kf = kernel_dft(w, 2, 2, 32, convention)
    for got, t in ((main, 4), (tail, 1)):
        want = np.zeros(1024, complex)
        for e in range(1024):
            kb, v, lane = e // 256, (e // 64) % 4, e % 64
            q, j = lane // 16, lane % 16
            row = 16 * (kb >> 1) + (q + 4 * v if form == "fp64" else 4 * q + v)
            want[e] = Kf[row, 16 * (kb & 1) + j] ** t / 1024
        assert np.abs(got - want).max() < 1e-15 * np.abs(want).max() * 8, t
        assert abs(got[0] - 1.3 ** t / 1024) < 1e-16  # K(0)^t = (sum w)^t
    plan.close()


def test_spectrum_heat1d_closed_form(ffs, torch_cuda):
    # 240-point prime-factor map: entry (v, lane) -> row frequency k0 = q + 4 v (< 15), column frequency
    # k1 = lane % 16, spectrum index k = (15 k1 + 16 k0) mod 240; Heat-1D: K^t = ((1 + cos th)/2)^t e^{-i th t}
    T, t = 40, 32
    plan = ffs.Plan(1, (5000,), np.array([0.25, 0.5, 0.25]), 1, T, precision="fp64", fuse=t)
    info = plan.info
    assert (info["fuse"], info["fuse_tail"]) == (t, T - t)
    main, tail = spectrum(plan, 256)
    for got, tt in ((main, t), (tail, T - t)):
        for e in range(256):
            v, lane = e // 64, e % 64
            k0, k1 = lane // 16 + 4 * v, lane % 16
            if k0 >= 15:
                assert got[e] == 0
                continue
            m = (15 * k1 + 16 * k0) % 240
            th = 2 * np.pi * m / 240
            want = ((1 + np.cos(th)) / 2) ** tt * np.exp(-2j * np.pi * ((m * tt) % 240) / 240) / 240
            assert abs(got[e] - want) < 1e-16, (e, tt)
    plan.close()


def test_spectrum_3d(ffs, torch_cuda):
    # entry (k2 block, reg v, lane): k0 = lane % 16, k1 = q + 4 v (FP64 order), k2 = block
    _, r, w, _ = ffs.named_stencil("Box3D27P", seed=7)
    plan = ffs.Plan(3, (40, 40, 40), w, r, 2, precision="fp64", fuse=2)
    main, _ = spectrum(plan, 4096)
    Kf = kernel_dft(w, 1, 3, 16, "ref")
    want = np.zeros(4096, complex)
    for e in range(4096):
        kb, v, lane = e // 256, (e // 64) % 4, e % 64
        want[e] = Kf[lane % 16, lane // 16 + 4 * v, kb] ** 2 / 4096
    assert np.abs(main - want).max() < 1e-15 * np.abs(want).max() * 8
    plan.close()


def test_read_table_errors(ffs, torch_cuda):
    _, r, w, _ = ffs.named_stencil("Box2D9P", seed=1)
    plan = ffs.Plan(2, (64, 64), w, r, 3, precision="fp64", tile=16)
    with pytest.raises(ffs.FFSError, match="UNSUPPORTED"):
        plan.read_table(1)  # no mixed operands in an FP64 plan
    with pytest.raises(ffs.FFSError, match="INVALID_ARG"):
        plan.read_table(9)
    plan.close()
    direct = ffs.Plan(2, (64, 64), w, r, 3, precision="fp64", algorithm="direct")
    with pytest.raises(ffs.FFSError, match="UNSUPPORTED"):
        direct.read_table(0)
    direct.close()


# ---- tables of the kernels that runs launch ----
LD = np.longdouble
PI = 4 * np.arctan(LD(1))


def trig(n, P):
    """cos and sin of pi (2a + 1)(2b + 1) / (2 P), a, b < n, in extended precision (exact angle reduction)."""
    k = 2 * np.arange(n) + 1
    th = PI * (np.outer(k, k) % (4 * P)).astype(LD) / (2 * P)
    return np.cos(th), np.sin(th)


def real_filter(L1, L2, P):
    """(alpha, beta, gamma, delta) of the window's filter from L(w0, w1) and L(w0, -w1), with the transforms' 4 / P^2."""
    s = LD(2) / (P * P)
    return np.stack([(L1.real + L2.real) * s, (L2.real - L1.real) * s, (L1.imag + L2.imag) * s, (L1.imag - L2.imag) * s], -1)


def half_sample_gain(w, K, convention, k0, k1, P, t):
    """(sum g[e] exp(i (w0 e0 + w1 e1)))^t and the same at -w1, w = pi (2k + 1) / P, correlation taps g."""
    g = np.asarray(w, dtype=LD).reshape(K, K)
    if convention == "ref":
        g = g[::-1, ::-1]
    e = np.arange(K)
    out = []
    for sign in (1, -1):
        L = np.zeros(k0.shape, dtype=np.clongdouble)
        for a in range(K):
            for b in range(K):
                m = ((2 * k0 + 1) * e[a] + sign * (2 * k1 + 1) * e[b]) % (2 * P)
                th = PI * m.astype(LD) / P
                L = L + g[a, b] * (np.cos(th) + 1j * np.sin(th))
        p = np.ones_like(L)
        for _ in range(t):
            p = p * L
        out.append(p)
    return out


def halves(words, f16):
    """The two 16-bit values of each 32-bit word, low half first, as numbers."""
    w = np.stack([words & 0xFFFF, words >> 16], -1).astype(np.uint32)
    return w.astype(np.uint16).view(np.float16).astype(LD) if f16 else (w << 16).view(np.float32).astype(LD)


def _matrix_gain():
    """The FP64 filters take out the gain of the matrices' rounding to doubles: a constant window through the rounded
    sine matrix and back, mean over the near half, both axes; the kernels' constant is 1.1e-16."""
    sine = trig(16, 32)[1].astype(np.float64).astype(LD)
    gain = float((sine.T @ (sine @ np.full(16, LD(2))) / 16).mean() - 1)
    assert abs(2 * gain - 1.1e-16) < 2e-17, gain
    return 1 - LD(1.1e-16)


MATRIX_GAIN = _matrix_gain()
LANES = np.arange(64)
Q, J = LANES // 16, LANES % 16


@pytest.mark.parametrize("convention", ["ref", "centred"])
@pytest.mark.parametrize("radius,fuse,tail", [(2, 4, 1), (1, 8, 5), (7, 1, 0)])
def test_real_tables_32_fp64(ffs, torch_cuda, convention, radius, fuse, tail):
    rng = np.random.default_rng(radius)
    K = 2 * radius + 1
    w = rng.standard_normal(K * K)
    w /= np.abs(w).sum()
    with ffs.Plan(2, (200, 200), w, radius, 2 * fuse + tail, fuse=fuse, tile=32, convention=convention) as plan:
        ops, filt = table(plan, 4, np.float64).reshape(2, 4, 64), table(plan, 5, np.float64)
    for got, want in zip(ops, trig(16, 32)):
        for v in range(4):  # lane (j + 16 k): entry (4 v + k, j)
            assert np.abs(got[v] - want[4 * v + Q, J]).max() <= 2.0 ** -53
    depths = [fuse] + ([tail] if tail else [])
    assert filt.size == 1024 * len(depths)
    for got, t in zip(filt.reshape(-1, 4, 64, 4), depths):
        for v in range(4):  # entry v * 64 + lane: (k0, k1) = (q + 4 v, j)
            want = MATRIX_GAIN * real_filter(*half_sample_gain(w, K, convention, Q + 4 * v, J, 32, t), 32)
            assert np.abs(got[v] - want).max() <= 2.0 ** -53 * np.abs(want).max()  # |entries| <= 2^-8 or so, rounded once


@pytest.mark.parametrize("convention", ["ref", "centred"])
@pytest.mark.parametrize("form", ["f16", "bf16"])
@pytest.mark.parametrize("radius,fuse,tail,gain", [(2, 4, 3, 1.0), (1, 8, 1, 0.25), (3, 3, 0, 1.7), (15, 1, 1, 0.5)])
def test_wide_tables(ffs, torch_cuda, convention, form, radius, fuse, tail, gain):
    rng = np.random.default_rng(radius)
    K = 2 * radius + 1
    w = rng.standard_normal(K * K)
    L = half_sample_gain(w, K, convention, *np.meshgrid(np.arange(32), np.arange(32), indexing="ij"), 64, 1)
    w *= gain / float(max(np.abs(x).max() for x in L))
    steps = 4 * fuse + tail
    with ffs.Plan(2, (100, 120), w, radius, steps, fuse=fuse, precision=form, convention=convention) as plan:
        assert plan.info["run_kernel"] == ffs.RUN_KERNELS["wide"]
        words, filt = table(plan, 4, np.uint32), table(plan, 5, np.float32).astype(LD)
    nt = 2 if form == "f16" else 3
    terms = halves(words.reshape(2, 2, nt, 64, 4), form == "f16").reshape(2, 2, nt, 64, 8).sum(axis=2)
    for got, want in zip(terms, trig(32, 64)):
        for b in range(2):
            for e in range(8):  # element e of lane (j + 16 q): entry (2 (4q + (e & 3)) + (e >> 2), 2j + b)
                err = np.abs(got[b, :, e] - want[2 * (4 * Q + (e & 3)) + (e >> 2), 2 * J + b]).max()
                assert err <= (2.0 ** -22 if form == "f16" else 2.0 ** -24)
    depths = [2 * fuse] + ([tail] if tail else [])
    assert filt.size == 4096 * len(depths)
    for got, t in zip(filt.reshape(-1, 4, 4, 64, 4), depths):
        scale = 1.0
        if form == "f16":  # normalised: |K|^t times a power of two in (1/2, 1] at its largest over the window's frequencies
            scale = 2.0 ** -np.ceil(t * np.log2(gain) - 1e-9)
            assert 0.5 < gain ** t * scale <= 1.0 + 1e-6
        for b in range(4):
            for v in range(4):  # entry (b * 4 + v) * 64 + lane: (2 (4q + v) + b0, 2j + b1)
                want = scale * real_filter(*half_sample_gain(w, K, convention, 2 * (4 * Q + v) + (b >> 1), 2 * J + (b & 1), 64, t), 64)
                assert np.abs(got[b, v] - want).max() <= 2.0 ** -23 * gain ** t * scale / 1024


@pytest.mark.parametrize("convention", ["ref", "centred"])
@pytest.mark.parametrize("form,radius,sizes,steps", [("fp64", 1, (150, 131, 139), 7), ("bf16", 1, (150, 131, 139), 7),
                                                     ("fp64", 2, (121, 113, 140), 3), ("bf16", 3, (90, 131, 157), 2)])
def test_stream_tables(ffs, torch_cuda, convention, form, radius, sizes, steps):
    K = 2 * radius + 1
    rng = np.random.default_rng(radius)
    w = rng.random(K ** 3)
    w /= w.sum()
    with ffs.Plan(3, sizes, w, radius, steps, precision=form, convention=convention) as plan:
        info = plan.info
        assert info["run_kernel"] == ffs.RUN_KERNELS["stream"]
        raw, filt = plan.read_table(4), table(plan, 5, np.float64 if form == "fp64" else np.float32).astype(LD)
    if form == "fp64":
        ops = np.frombuffer(raw, np.float64).reshape(2, 4, 64)
        for got, want in zip(ops, trig(16, 32)):
            for v in range(4):
                assert np.abs(got[v] - want[4 * v + Q, J]).max() <= 2.0 ** -53
    else:  # pairings (h|h), (m|m), (l|h): elements 0..3 of the three hold the terms, 4..7 their partners
        ops = halves(np.frombuffer(raw, np.uint32).reshape(2, 3, 64, 4), False).reshape(2, 3, 64, 8)
        for got, want in zip(ops, trig(16, 32)):
            for e in range(4):
                assert np.abs(got[:, :, e].sum(axis=0) - want[4 * Q + e, J]).max() <= 2.0 ** -24
                assert np.array_equal(got[:, :, e + 4], got[[0, 1, 0], :, e])
    depths = [info["run_depth"]] + ([steps % info["run_depth"]] if steps % info["run_depth"] else [])
    E = 2 * radius * info["run_depth"] + 1
    g = np.asarray(w, dtype=LD).reshape(K, K, K)
    if convention == "ref":
        g = g[::-1, ::-1, ::-1]
    for got, t in zip(filt.reshape(len(depths), E, 4, 64, 4), depths):
        for v in range(4):
            k1 = 4 * Q + v if form == "bf16" else Q + 4 * v
            poly = [np.zeros((E, 64), dtype=np.clongdouble) for _ in range(2)]
            for p in poly:
                p[0] = 1
            one = [np.zeros((K, 64), dtype=np.clongdouble) for _ in range(2)]
            for s, sign in enumerate((1, -1)):
                for a in range(K):
                    for b in range(K):
                        for c in range(K):
                            th = PI * (((2 * k1 + 1) * b + sign * (2 * J + 1) * c) % 64).astype(LD) / 32
                            one[s][a] += g[a, b, c] * (np.cos(th) + 1j * np.sin(th))
                for _ in range(t):
                    nxt = np.zeros_like(poly[s])
                    for i in range(E):
                        for a in range(K):
                            if i + a < E:
                                nxt[i + a] += poly[s][i] * one[s][a]
                    poly[s] = nxt
            for e in range(E):
                want = real_filter(poly[0][e], poly[1][e], 32) * (MATRIX_GAIN if form == "fp64" else 1)
                assert np.abs(got[e, v] - want).max() <= (2.0 ** -52 if form == "fp64" else 2.0 ** -24) * np.abs(want).max() + 1e-300


@pytest.mark.parametrize("convention", ["ref", "centred"])
@pytest.mark.parametrize("form,algorithm,radius,n,steps", [("fp64", "fft", 3, 900, 101), ("fp64", "direct", 1, 5000, 248),
                                                           ("bf16", "fft", 3, 900, 101), ("bf16", "fft", 60, 2000, 9)])
def test_line_tables(ffs, torch_cuda, convention, form, algorithm, radius, n, steps):
    K = 2 * radius + 1
    rng = np.random.default_rng(radius)
    w = rng.standard_normal(K)
    w /= np.abs(w).sum()
    with ffs.Plan(1, (n,), w, radius, steps, precision=form, algorithm=algorithm, convention=convention) as plan:
        info = plan.info
        assert info["run_kernel"] == ffs.RUN_KERNELS["line"]
        taps = table(plan, 5, np.float64).reshape(-1, 512)
        words = table(plan, 4, np.uint32) if form == "bf16" else None
    depths = [info["run_depth"]] + ([steps % info["run_depth"]] if steps % info["run_depth"] else [])
    assert len(taps) == len(depths)
    for d, (got, t) in enumerate(zip(taps, depths)):
        one = np.asarray(w, dtype=LD)[::-1 if convention == "ref" else 1]
        powers = [np.array([1], dtype=LD)]
        for _ in range(t):
            powers.append(np.convolve(powers[-1], one))
        g, h = powers[t], np.abs(powers[t // 2])
        # rounded once, and for more than 128 taps the two halves of the last square (and the odd step's factor) before it
        halves_of = np.convolve(h, h) if t % 2 == 0 else np.convolve(np.convolve(h, h), np.abs(one))
        bound = 2.0 ** -53 * (np.abs(g) + (3 * halves_of if g.size > 128 else 0)).max()
        assert np.abs(got[:g.size] - g).max() <= bound * (1 + 1e-9) and not got[g.size:].any()
        if words is None:
            continue
        T = halves(words.reshape(len(depths), -1, 3, 64, 4)[d], False).reshape(-1, 3, 64, 8).sum(axis=1)
        pad = np.concatenate([np.zeros(16, LD), g, np.zeros(32 * len(T) + 16, LD)])
        for b in range(len(T)):
            for e in range(8):  # element e of lane (i + 16 q): T[i][32 b + 8 q + e] = g[32 b + 8 q + e - i]
                k = 32 * b + 8 * Q + e - J
                want = np.where(k >= 0, pad[np.maximum(k, 0) + 16], 0)
                assert np.abs(T[b, :, e] - want).max() <= 2.0 ** -24 * np.abs(g).max()
    if form == "fp64":
        with ffs.Plan(1, (n,), w, radius, steps, precision=form, algorithm=algorithm, convention=convention) as plan:
            with pytest.raises(ffs.FFSError, match="UNSUPPORTED"):
                plan.read_table(4)  # the FP64 product reads the taps themselves
