"""The split-bf16 GEMM (gemm_sbf.hip, M > 8, every weight format) against 64-bit products.

Every operand is split exactly into bf16 terms and the products of the terms
that matter are summed in fp32, so an output differs from the 64-bit product
of the same operands by at most one fp32 rounding of each 32-deep slice's sum,
the small terms, dropped (at most 2^-24 of a product together) or summed apart, and
the epilogue's own roundings:
    |C - ref| <= (ceil(K / 32) + 8) * 2^-24 * sum_k |a b| + 2^-23 |ref|.
Outputs the split does not carry (infinities, NaNs, values past the largest
bf16, sums that elements below 2^-102 or products below 2^-80 may have put off) are
recomputed in fp32, as the reference sums (src/core/ops.zig:277-414), so their inf /
NaN pattern is the oracle's.  Int8 / int4 weights take two terms of A (|x - hi - lo| <= 2^-17 |x|) and
share one sum, which a slice rounds twice:
    |C - ref| <= (2^-17 + (2 ceil(K / 32) + 8) * 2^-24) * sum_k |a b| + 2^-23 |ref|.
A K split adds one rounding a split.  TML_GEMM_SBF_TILE / _SPLIT pick a tile and
a K split, TML_GEMM_SBF=0 turns the kernel off.
"""
import os

import numpy as np
import pytest

from tomoul_amd import _abi, synth

pytestmark = pytest.mark.gpu
TILES = (1, 2, 3, 4, 5)


@pytest.fixture
def env():
    keys = ("TML_GEMM_SBF_TILE", "TML_GEMM_SBF_SPLIT", "TML_GEMM_SBF", "TML_REQUIRE_SPLIT")
    saved = {key: os.environ.get(key) for key in keys}
    yield os.environ
    for key, v in saved.items():
        if v is None:
            os.environ.pop(key, None)
        else:
            os.environ[key] = v


def weight(orc, fmt, w):
    """(bytes, scales, the fp32 values [K,N]) of w in format fmt."""
    if fmt == _abi.FMT_F32:
        return w, None, w
    if fmt == _abi.FMT_F16:
        h = orc.to_f16(w)
        return h, None, h.view(np.float16).astype(np.float32).reshape(w.shape)
    q, s = orc.quantize_q8k(w)
    flat = np.repeat(s, 32)[: w.size] * q.reshape(-1).astype(np.float32)
    return q, s, flat.astype(np.float32).reshape(w.shape)


def run(fmt, m, n, k, a, q, scales, **kw):
    c = np.zeros((m, n), np.float32)
    _abi.gemm(fmt, m, n, k, a, np.ascontiguousarray(q), c, scales=scales, **kw)
    return c


def check(c, a, w, bias=None, res=None, terms=3):
    ref = a.astype(np.float64) @ w.astype(np.float64)
    mag = np.abs(a).astype(np.float64) @ np.abs(w).astype(np.float64)
    slices = -(-a.shape[1] // 32)
    bound = ((slices + 8) * 2.0**-24 if terms == 3 else 2.0**-17 + (2 * slices + 8) * 2.0**-24) * mag
    for x in (bias, res):
        if x is not None:
            ref = ref + x
            bound = bound + 2.0**-24 * (np.abs(ref) + np.abs(x))
    worst = float(np.max(np.abs(c - ref) / (bound + 2.0**-23 * np.abs(ref) + 1e-300)))
    assert worst <= 1.0, worst


@pytest.mark.parametrize("fmt", [_abi.FMT_F32, _abi.FMT_F16, _abi.FMT_Q8_K])
@pytest.mark.parametrize("tile", TILES)
def test_sbf_tiles(orc, env, tile, fmt):
    # partial tiles in M and N, one slice to many, K not a whole slice
    env["TML_GEMM_SBF_TILE"] = str(tile)
    for (m, n, k) in [(9, 32, 4), (33, 160, 36), (257, 288, 520), (130, 96, 1032)]:
        if fmt != _abi.FMT_Q8_K:
            n += 1  # odd rows: the scalar stores, unaligned B rows
        a, bias = synth.normal_matrix(11 + m, m, k), synth.normal(12, n, 0.0, 0.02)
        q, scales, w = weight(orc, fmt, synth.normal_matrix(13, k, n, 0.02))
        check(run(fmt, m, n, k, a, q, scales, bias=bias), a, w, bias.astype(np.float64))


@pytest.mark.parametrize("fmt,m,n,k", [(_abi.FMT_F32, 300, 5120, 1280), (_abi.FMT_F16, 700, 2048, 640),
                                       (_abi.FMT_Q8_K, 900, 3072, 768), (_abi.FMT_F32, 77, 1001, 388)])
def test_sbf_default_plan_epilogue(orc, fmt, m, n, k):
    # the planner's own choice, with the residual and both activations
    a, bias, res = synth.normal_matrix(21, m, k), synth.normal(22, n, 0.0, 0.02), synth.normal_matrix(23, m, n)
    q, scales, w = weight(orc, fmt, synth.normal_matrix(24, k, n, 0.02))
    c = np.zeros((m, n), np.float32)
    _abi.gemm_residual(fmt, m, n, k, a, q, res, c, scales=scales, bias=bias)
    check(c, a, w, bias.astype(np.float64), res.astype(np.float64))
    plain = run(fmt, m, n, k, a, q, scales, bias=bias)
    for act, gelu in ((_abi.ACT_GELU_ERF, orc.gelu_exact), (_abi.ACT_GELU_TANH, orc.gelu_tanh)):
        _abi.gemm_act(fmt, m, n, k, a, q, c, act=act, scales=scales, bias=bias)
        ref = gelu(plain)
        assert np.max(np.abs(c - ref)) <= 1e-6 * max(1.0, np.max(np.abs(ref))), act


@pytest.mark.parametrize("fmt", [_abi.FMT_F32, _abi.FMT_F16, _abi.FMT_Q8_K])
@pytest.mark.parametrize("tile,split", [(t, 1) for t in TILES] + [(3, 2), (5, 3)])
def test_sbf_any_k(orc, env, tile, split, fmt):
    # K of no whole 16-byte load: rows of A start on any dword, and the last row's
    # last load crosses the end of A
    env["TML_GEMM_SBF_TILE"], env["TML_GEMM_SBF_SPLIT"] = str(tile), str(split)
    for (m, n, k) in [(9, 32, 1), (33, 160, 35), (257, 288, 518), (130, 96, 1033)]:
        a, bias = synth.normal_matrix(81 + m, m, k), synth.normal(82, n, 0.0, 0.02)
        q, scales, w = weight(orc, fmt, synth.normal_matrix(83, k, n, 0.02))
        check(run(fmt, m, n, k, a, q, scales, bias=bias), a, w, bias.astype(np.float64))


def test_sbf_unaligned_a():
    # A on any dword, K odd or even, the planner's own choice
    import torch
    for (m, n, k, off) in [(40, 130, 255, 1), (300, 512, 256, 2), (77, 97, 1030, 3)]:
        gen = torch.Generator(device="cuda").manual_seed(k)
        flat = torch.randn(m * k + off, generator=gen, device="cuda")
        a, w = flat[off:].reshape(m, k), torch.randn(k, n, generator=gen, device="cuda") * 0.02
        c = torch.zeros(m, n, device="cuda")
        _abi.gemm_dev(_abi.FMT_F32, m, n, k, a.data_ptr(), w.data_ptr(), c.data_ptr(),
                      stream=torch.cuda.current_stream().cuda_stream)
        check(c.cpu().numpy(), a.cpu().numpy(), w.cpu().numpy())


@pytest.mark.parametrize("tile", TILES)
def test_sbf_inf_nan(orc, env, tile):
    env["TML_GEMM_SBF_TILE"] = str(tile)
    m, n, k = 140, 100, 100  # K is no whole slice: row r's tail reads row r + 1's head
    a, w = synth.normal_matrix(31, m, k), synth.normal_matrix(32, k, n, 0.02)
    a[3, 5], a[4, 0], a[64, 99], a[139, 7] = np.inf, -np.inf, np.nan, np.float32(3.4028235e38)
    w[5, 9], w[7, 10], w[11, 20], w[12, 21] = 0.0, 0.0, np.inf, np.nan
    a[70, 11] = 0.0
    c, ref = run(_abi.FMT_F32, m, n, k, a, w, None), orc.matmul(a, w)
    assert np.array_equal(np.isnan(c), np.isnan(ref)) and np.array_equal(np.isposinf(c), np.isposinf(ref))
    assert np.array_equal(np.isneginf(c), np.isneginf(ref))
    fin = np.isfinite(ref)
    # the recomputed sums and the others alike, 100 terms
    mag = np.where(np.isfinite(a), np.abs(a), 0).astype(np.float64) @ np.where(np.isfinite(w), np.abs(w), 0)
    assert np.all(np.abs(c[fin].astype(np.float64) - ref[fin]) <= 2.0**-23 * 100 * mag[fin])


@pytest.mark.parametrize("scale", [2.0**-100, 2.0**-60, 2.0**60, 2.0**110])
def test_sbf_range(env, scale):
    # the whole exponent range of A: a power of two times the operand is the same
    # power times the result, also where the third term falls under bf16's
    # denormals (there the sum is recomputed in fp32: K roundings)
    env["TML_GEMM_SBF_TILE"] = "5"
    m, n, k = 70, 65, 96
    a, w = synth.normal_matrix(41, m, k), synth.normal_matrix(42, k, n, 0.02)
    c = run(_abi.FMT_F32, m, n, k, a * np.float32(scale), w, None).astype(np.float64) / scale
    ref = a.astype(np.float64) @ w.astype(np.float64)
    mag = np.abs(a).astype(np.float64) @ np.abs(w).astype(np.float64)
    assert np.max(np.abs(c - ref) / mag) <= k * 2.0**-24


SMALL = [(-115, 60), (-120, 60), (-125, 70), (-130, 90), (-135, 21), (-140, 100), (60, -120), (90, -130), (100, -140)]


@pytest.mark.parametrize("tile,split", [(t, 1) for t in TILES] + [(3, 2), (5, 3)])
@pytest.mark.parametrize("ea,eb", SMALL)
def test_sbf_small_operands(env, tile, split, ea, eb):
    """Operands whose terms reach bf16's denormals, or have none (below 2^-134),
    against large ones: fp32 precision, K roundings at most, as the fp32 matrix cores give."""
    env["TML_GEMM_SBF_TILE"], env["TML_GEMM_SBF_SPLIT"] = str(tile), str(split)
    m, n, k = 140, 101, 130
    a, w = np.ldexp(synth.normal_matrix(101, m, k), ea), np.ldexp(synth.normal_matrix(102, k, n), eb)
    a[7] = 0.0  # a sum of zeros
    w[:, 9] = 0.0
    a[11, 1::2], w[1::2, 12] = -a[11, ::2], w[::2, 12]  # and of values that cancel
    # row 70 tiny among ordinary values, one large column: only their own outputs are in doubt
    a[70], w[:, 70] = np.ldexp(a[70], -ea - 125), np.ldexp(w[:, 70], 20 - eb)  # (2^20: the large products stay finite)
    c = run(_abi.FMT_F32, m, n, k, a, w, None).astype(np.float64)
    ref = a.astype(np.float64) @ w.astype(np.float64)
    mag = np.abs(a).astype(np.float64) @ np.abs(w).astype(np.float64)
    # (2^-149 a product where the fp32 products themselves are denormal)
    bound = k * 2.0**-24 * mag + np.where(mag < 2.0**-100, k * 2.0**-149, 0.0)
    assert np.all(np.abs(c - ref) <= bound), float(np.max(np.abs(c - ref) / (mag + 1e-300)))


@pytest.mark.parametrize("tile", [2, 3, 5])
@pytest.mark.parametrize("fmt,ea,ew", [(_abi.FMT_F16, -138, 12), (_abi.FMT_Q8_K, -125, 60), (_abi.FMT_Q8_K, 90, -130),
                                       (_abi.FMT_Q8_0, -138, 0)])
def test_sbf_small_operands_formats(orc, env, tile, fmt, ea, ew):
    # the same with f16, Q8_K and (odd N: three terms) int8 weights
    env["TML_GEMM_SBF_TILE"] = str(tile)
    m, n, k = 140, 96 if fmt == _abi.FMT_Q8_K else 97, 130
    a, scale = np.ldexp(synth.normal_matrix(103, m, k), ea), 1.0
    raw = synth.normal_matrix(104, k, n)
    if fmt == _abi.FMT_Q8_0:
        (q, _), scales, scale = orc.quantize_q8(raw), None, 2.0**20
        w = q.reshape(k, n).astype(np.float64) * scale
    else:
        q, scales, w = weight(orc, fmt, np.ldexp(raw, ew))
    c = np.zeros((m, n), np.float32)
    _abi.gemm(fmt, m, n, k, a, np.ascontiguousarray(q), c, scale=scale, scales=scales)
    ref = a.astype(np.float64) @ w.astype(np.float64)
    mag = np.abs(a).astype(np.float64) @ np.abs(w).astype(np.float64)
    assert np.all(np.abs(c - ref) <= k * 2.0**-24 * mag), float(np.max(np.abs(c - ref) / mag))


@pytest.mark.parametrize("tile,split", [(t, 1) for t in TILES] + [(3, 2), (5, 3)])
@pytest.mark.parametrize("k", [128, 100])
def test_sbf_zero_rows(env, tile, split, k):
    # rows of zeros between others (k = 100: the last slice reads on into the next row):
    # zeros, a NaN where the weight is infinite, and a zero where it is past the largest bf16;
    # a row of zeros and one NaN
    env["TML_GEMM_SBF_TILE"], env["TML_GEMM_SBF_SPLIT"] = str(tile), str(split)
    m, n = 140, 101
    a, w = synth.normal_matrix(131, m, k), synth.normal_matrix(132, k, n, 0.02)
    zero = np.r_[2, 17:40, 63, 64, 100:140]
    a[zero] = 0.0
    a[17, 3] = np.nan
    w[5, 9], w[k - 1, 50], w[:, 70] = np.inf, np.float32(3.4028235e38), 0.0
    c = run(_abi.FMT_F32, m, n, k, a, w, None)
    with np.errstate(invalid="ignore", over="ignore"):  # (column 50 overflows fp32 where |a| > 1)
        ref = (a.astype(np.float64) @ w.astype(np.float64)).astype(np.float32)
    assert np.array_equal(np.isnan(c), np.isnan(ref)) and np.array_equal(np.isinf(c), np.isinf(ref))
    rows = np.isfinite(a).all(1)
    assert np.all(c[zero][rows[zero]][:, np.arange(n) != 9] == 0.0) and np.all(c[rows][:, 70] == 0.0)
    cols = ~np.isin(np.arange(n), (9, 50))
    check(c[rows][:, cols], a[rows], w[:, cols])


def test_sbf_exact_integers(env):
    # products and sums of small integers are exact
    rng = np.random.default_rng(5)
    a, w = rng.integers(-999, 1000, (200, 320)).astype(np.float32), rng.integers(-9, 10, (320, 129)).astype(np.float32)
    for tile in TILES:
        env["TML_GEMM_SBF_TILE"] = str(tile)
        assert np.array_equal(run(_abi.FMT_F32, 200, 129, 320, a, w, None), a @ w)


@pytest.mark.parametrize("split", [2, 3])
@pytest.mark.parametrize("tile", TILES)
def test_sbf_split(env, tile, split):
    # raw partials of K splits (the last one short), added in split order by the
    # reduce launch with bias and residual; odd N takes the scalar partial stores
    env["TML_GEMM_SBF_TILE"], env["TML_GEMM_SBF_SPLIT"], env["TML_REQUIRE_SPLIT"] = str(tile), str(split), "1"
    for (m, n, k) in [(130, 97, 516), (257, 200, 260)]:
        a, bias, res = synth.normal_matrix(51, m, k), synth.normal(52, n, 0.0, 0.02), synth.normal_matrix(53, m, n)
        w = synth.normal_matrix(54, k, n, 0.02)
        c = np.zeros((m, n), np.float32)
        _abi.gemm_residual(_abi.FMT_F32, m, n, k, a, w, res, c, bias=bias)
        check(c, a, w, bias.astype(np.float64), res.astype(np.float64))


@pytest.mark.parametrize("tile,split", [(1, 1), (1, 3), (2, 1), (2, 2)])
def test_sbf_int(orc, env, tile, split):
    env["TML_GEMM_SBF_TILE"], env["TML_GEMM_SBF_SPLIT"] = str(tile), str(split)
    for (m, n, k) in [(9, 34, 40), (300, 130, 520), (257, 98, 1288)]:
        a, bias = synth.normal_matrix(61 + m, m, k), synth.normal(62, n, 0.0, 0.02)
        w = synth.normal_matrix(63, k, n, 0.02)
        q, s = orc.quantize_q8(w)
        p, s4 = orc.quantize_q4(w)
        qc, sc = orc.quantize_q8_cols(w)
        pc, sc4 = orc.quantize_q4_cols(w)
        for fmt, b, scale, scales, deq in [
                (_abi.FMT_Q8_0, q, s, None, orc.dequantize_q8(q, s)),
                (_abi.FMT_Q4_0, p, s4, None, orc.dequantize_q4(p, k * n, s4)),
                (_abi.FMT_Q8_0_PC, qc, 1.0, sc, orc.dequantize_cols(_abi.FMT_Q8_0_PC, qc, sc, k, n)),
                (_abi.FMT_Q4_0_PC, pc, 1.0, sc4, orc.dequantize_cols(_abi.FMT_Q4_0_PC, pc, sc4, k, n))]:
            c = run(fmt, m, n, k, a, b, scales, scale=scale, bias=bias)
            check(c, a, np.asarray(deq, np.float32).reshape(k, n), bias.astype(np.float64), terms=2)


@pytest.mark.parametrize("tile,split", [(0, 1), (2, 1), (3, 1), (3, 2), (5, 1), (5, 3)])
def test_sbf_int_exact(orc, env, tile, split):
    # int8 / int4 outside gemm_qbf.hip's layouts (odd N, K % 8 != 0): three terms of
    # A, within the fp32 products' bound; 0: the planner's own choice
    if tile:
        env["TML_GEMM_SBF_TILE"], env["TML_GEMM_SBF_SPLIT"] = str(tile), str(split)
    for (m, n, k) in [(9, 33, 5), (300, 130, 517), (257, 97, 1288), (70, 64, 1026)]:
        a, bias = synth.normal_matrix(91 + m, m, k), synth.normal(92, n, 0.0, 0.02)
        w = synth.normal_matrix(93, k, n, 0.02)
        q, s = orc.quantize_q8(w)
        qc, sc = orc.quantize_q8_cols(w)
        check(run(_abi.FMT_Q8_0, m, n, k, a, q, None, scale=s, bias=bias), a, orc.dequantize_q8(q, s).reshape(k, n),
              bias.astype(np.float64))
        check(run(_abi.FMT_Q8_0_PC, m, n, k, a, qc, sc, bias=bias), a,
              np.asarray(orc.dequantize_cols(_abi.FMT_Q8_0_PC, qc, sc, k, n), np.float32).reshape(k, n),
              bias.astype(np.float64))
        if n % 2 == 0:
            p, s4 = orc.quantize_q4(w)
            check(run(_abi.FMT_Q4_0, m, n, k, a, p, None, scale=s4, bias=bias), a,
                  orc.dequantize_q4(p, k * n, s4).reshape(k, n), bias.astype(np.float64))


@pytest.mark.parametrize("fmt", [_abi.FMT_Q8_0, _abi.FMT_Q4_0])
@pytest.mark.parametrize("m,n,k", [(1500, 1536, 388), (600, 1000, 1028), (20, 1000, 132)])
def test_sbf_int_k4(orc, fmt, m, n, k):
    # K % 8 == 4 with wide loads, the planner's own choice: the split-bf16 kernel at the
    # largest, the fp32-MFMA kernels (600 x 1000 has few tiles) at the others
    a, bias, w = synth.normal_matrix(121, m, k), synth.normal(122, n, 0.0, 0.02), synth.normal_matrix(123, k, n, 0.02)
    q, s = (orc.quantize_q8 if fmt == _abi.FMT_Q8_0 else orc.quantize_q4)(w)
    deq = (orc.dequantize_q8(q, s) if fmt == _abi.FMT_Q8_0 else orc.dequantize_q4(q, k * n, s)).reshape(k, n)
    c = run(fmt, m, n, k, a, q, None, scale=s, bias=bias)
    ref = a.astype(np.float64) @ deq.astype(np.float64) + bias
    # 2-norm: 0.6e-7 - 2.8e-7 on the split kernel, up to 9.9e-7 on the fp32 matrix cores
    assert np.linalg.norm(c - ref) <= (3e-7 if m == 1500 else 1e-6) * np.linalg.norm(ref)


@pytest.mark.parametrize("tile", [1, 2])
def test_sbf_int_inf_nan(orc, env, tile):
    env["TML_GEMM_SBF_TILE"] = str(tile)
    m, n, k = 140, 100, 72
    a = synth.normal_matrix(71, m, k)
    a[3, 5], a[4, 0], a[64, 71], a[139, 7] = np.inf, -np.inf, np.nan, np.float32(3.4028235e38)
    q, s = orc.quantize_q8(synth.normal_matrix(72, k, n, 0.02))
    q = q.reshape(k, n).copy()
    q[7] = np.clip(q[7], -1, 1)  # FLT_MAX times these stays finite
    q[5, ::7] = 0
    c, ref = run(_abi.FMT_Q8_0, m, n, k, a, q, None, scale=s), orc.matmul_q8(a, q, s)
    assert np.array_equal(np.isnan(c), np.isnan(ref)) and np.array_equal(np.isinf(c), np.isinf(ref))
    fin = np.isfinite(ref)
    mag = np.where(np.isfinite(a), np.abs(a), 0).astype(np.float64) @ np.abs(q.astype(np.float64) * s)
    assert np.all(np.abs(c[fin].astype(np.float64) - ref[fin]) <= (2.0**-17 + 2.0**-23 * k) * mag[fin])


@pytest.mark.parametrize("split", [1, 2])
@pytest.mark.parametrize("fmt,n,k,tile", [(_abi.FMT_F32, 101, 101, 1), (_abi.FMT_F32, 101, 101, 4), (_abi.FMT_F16, 101, 101, 2),
                                          (_abi.FMT_F16, 101, 101, 5), (_abi.FMT_Q8_K, 160, 101, 2),
                                          (_abi.FMT_Q8_K, 160, 101, 3), (_abi.FMT_Q8_0, 104, 136, 1),
                                          (_abi.FMT_Q4_0, 98, 136, 1), (_abi.FMT_Q4_0, 98, 136, 2),
                                          (_abi.FMT_Q8_0, 101, 101, 2), (_abi.FMT_Q8_0, 101, 101, 5),
                                          (_abi.FMT_Q4_0, 98, 101, 3)])
def test_sbf_recomputed(orc, env, fmt, n, k, tile, split):
    # rows, columns and single elements that are not finite, every format on both
    # its arithmetics (k = 136: two terms of A, n odd or k = 101: three), with and without a
    # K split: the 64-bit product's pattern, and fp32 sums of K products elsewhere
    env["TML_GEMM_SBF_TILE"], env["TML_GEMM_SBF_SPLIT"] = str(tile), str(split)
    m, scale, scales = 140, 1.0, None
    a, raw = synth.normal_matrix(111, m, k), synth.normal_matrix(112, k, n, 0.02)
    a[3, 5], a[4, 0], a[31, 70], a[64, k - 1], a[90], a[139, 7] = np.inf, -np.inf, np.nan, np.inf, np.nan, np.inf
    raw[5, ::7], raw[70, 1::5] = 0.0, 0.0
    if fmt == _abi.FMT_F32:
        raw[11, 20], raw[12, 21], raw[:, 40] = np.inf, np.nan, -np.inf
    if fmt == _abi.FMT_Q8_0:
        (q, scale), terms = orc.quantize_q8(raw), 2 if k % 8 == 0 and n % 8 == 0 else 3
        w = orc.dequantize_q8(q, scale).reshape(k, n)
    elif fmt == _abi.FMT_Q4_0:
        (q, scale), terms = orc.quantize_q4(raw), 2 if k % 8 == 0 else 3
        w = orc.dequantize_q4(q, k * n, scale).reshape(k, n)
    else:
        (q, scales, w), terms = weight(orc, fmt, raw), 3
    if fmt == _abi.FMT_Q8_K:
        scales = scales.copy()
        scales[5 * n // 32 + 1] = np.nan  # 32 elements of row 5
        w[5, 32:64] = np.nan
    c = np.zeros((m, n), np.float32)
    _abi.gemm(fmt, m, n, k, a, np.ascontiguousarray(q), c, scale=scale, scales=scales)
    with np.errstate(invalid="ignore"):
        ref = a.astype(np.float64) @ w.astype(np.float64)
        assert np.array_equal(np.isnan(c), np.isnan(ref))
        assert np.array_equal(np.isposinf(c), np.isposinf(ref)) and np.array_equal(np.isneginf(c), np.isneginf(ref))
    fin, zero = np.isfinite(ref), lambda x: np.where(np.isfinite(x), np.abs(x), 0).astype(np.float64)
    bound = (k * 2.0**-24 + (2.0**-17 if terms == 2 else 0.0)) * (zero(a) @ zero(w)) + 2.0**-22 * np.abs(np.where(fin, ref, 0))
    assert np.all(np.abs(c - np.where(fin, ref, 0))[fin] <= bound[fin])


def test_sbf_split_plan_without_workspace(env):
    """512 x 1024 x 4096 in f32 splits K by default; a first call under stream
    capture, where the workspace cannot grow, runs an unsplit plan instead of
    being refused, and the allocation-free call serves the split one."""
    import torch
    torch.cuda.synchronize()
    _abi.shutdown()  # a fresh context has no workspace
    _abi.init()
    m, n, k = 512, 1024, 4096
    gen = torch.Generator(device="cuda").manual_seed(9)
    a, b = torch.randn(m, k, generator=gen, device="cuda"), torch.randn(k, n, generator=gen, device="cuda") * 0.02
    c = [torch.zeros(m, n, device="cuda") for _ in range(3)]
    ref = (a.double() @ b.double())
    side, g = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g, stream=side):
        _abi.gemm_dev(_abi.FMT_F32, m, n, k, a.data_ptr(), b.data_ptr(), c[0].data_ptr(), stream=side.cuda_stream)
    env["TML_REQUIRE_SPLIT"] = "1"
    _abi.gemm_ex_dev_noalloc(_abi.FMT_F32, m, n, k, a.data_ptr(), b.data_ptr(), c[1].data_ptr())
    _abi.gemm_dev(_abi.FMT_F32, m, n, k, a.data_ptr(), b.data_ptr(), c[2].data_ptr())
    for _ in range(3):
        c[0].zero_()
        g.replay()
        torch.cuda.synchronize()
        for x in c:
            assert float((x - ref).norm() / ref.norm()) <= 2e-6
    assert torch.equal(c[1], c[2])
