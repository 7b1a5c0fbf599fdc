"""The bounds stated for the bf16 split of the larger GEMMs (gemm_sbf.hip), over
every mantissa: an fp32 value is three bf16 terms exactly, |m| <= 2^-8 |x| and
|l| <= 2^-17 |x|; the dropped products ml + lm + ll are at most 2^-24 of a product, lm
for an f16 weight (two terms) 2^-25; two terms leave at most 2^-17 |x|."""
import numpy as np


def bf16(x):  # round to nearest even
    u = x.view(np.uint32)
    return ((u + np.uint32(0x7FFF) + ((u >> np.uint32(16)) & np.uint32(1))) & np.uint32(0xFFFF0000)).view(np.float32)


def terms(x):
    h = bf16(x)
    m = bf16(x - h)
    return h, m, x - h - m


def test_split_bounds():
    x = (np.arange(1 << 23, dtype=np.uint32) | np.uint32(0x3F800000)).view(np.float32)
    _, m, low = terms(x)
    assert np.array_equal(bf16(low), low)  # the third term is the rest, exactly
    rm, rl = np.abs(m) / x.astype(np.float64), np.abs(low) / x.astype(np.float64)
    assert 2.0**-8.01 < rm.max() <= 2.0**-8 and 2.0**-17.01 < rl.max() <= 2.0**-17
    # the largest m l pairs; ll adds 2^-34
    top = np.argsort(-rm * rl)[:200]
    dropped = np.max(rm[top][:, None] * rl[top] + rl[top][:, None] * rm[top] + rl[top][:, None] * rl[top])
    assert 2.0**-24.02 < dropped <= 2.0**-24
    # f16 weights, eleven bits: two terms, exactly
    y = ((np.arange(1 << 10, dtype=np.uint32) << np.uint32(13)) | np.uint32(0x3F800000)).view(np.float32)
    _, my, ly = terms(y)
    assert not ly.any() and np.max(np.abs(my) / y) * rl.max() <= 2.0**-25
