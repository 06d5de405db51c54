"""The bound on the matrix-core estimate of a rotated channel (PolarQuant codes,
turboquant_pro/core.py:542-617), restated in NumPy: the kernel's bound covers
every MFMA that it issues, and the estimate with every addend truncated at the
accumulator's scale stays within it, for rows of the lengths that the estimate
takes; at row length 1e-6, which it leaves to the ordered sum, it does not."""

import os
import re

import numpy as np
import pytest

from oracle import tq_oracle as O

f16, f32, f64 = np.float16, np.float32, np.float64
HEADER = open(os.path.join(os.path.dirname(__file__), "..", "turboquant-pro_amd", "csrc", "tqk_common.h")).read()


def _bound():
    m = re.search(r"kEstimateBound = ([\d.]+)f;", HEADER)
    assert m and "kEstimateBound * (float)D * 0x1p-22f * __builtin_sqrtf(most)" in HEADER
    return float(m.group(1))


def _mfmas(lo):
    """MFMAs per 32 channels and 16 x 16 tile: those of low halves, and after all of them those of high ones."""
    body = HEADER[HEADER.index("void polar_codes("):HEADER.index("void set_code(")]
    loops = [x for x in re.split(r"for \(int ks = 0; ks < D / 32; \+\+ks\)", body)[1:]]
    assert len(loops) == 2 and body.count("__builtin_amdgcn_mfma") == 2   # (one of the two operand orders)
    first, second = loops[0], loops[1].split(";")[0]
    low = first.count("add(row + 32 * ks, pf.lo[ks])") + lo * first.count("if constexpr (LO) add(row + D + 32 * ks, pf.hi[ks])")
    assert first.count("add(") == 2 and second.strip() == "add(row + 32 * ks, pf.hi[ks])"
    return low, 1


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("lo", [False, True], ids=["fp16", "fp32"])
def test_bound_counts_every_mfma(D, lo):
    low, high = _mfmas(lo)
    assert (low, high) == ((2, 1) if lo else (1, 1))
    ordered = D * 2.0 ** -24
    mfma = (D / 32) * 33 * 2.0 ** -23 * (high + 2.0 ** -10 * low)
    rest = 3 * 2.0 ** -22 + 2.0 ** -22 + D ** 0.5 * 2.0 ** -33 / 2.0 ** -8
    assert ordered + mfma + rest <= 0.99 * _bound() * D * 2.0 ** -22   # 0.99: |u| and N themselves are rounded


def _pair(x):
    h = x.astype(f16)
    return h.astype(f64), (x - h.astype(f32)).astype(f16).astype(f64)


def _mfma(acc, a, b):
    """acc + sum over 32 channels of a b, every addend cut to 24 bits at the largest one's scale."""
    add = np.concatenate([acc[..., None], a[:, None, :] * b[None, :, :]], axis=2)
    big = np.abs(add).max(axis=2, keepdims=True)
    step = np.exp2(np.floor(np.log2(np.where(big > 0, big, 1.0))) - 23)
    return np.trunc(add / step).sum(axis=2) * step[..., 0]


def _worst(D, lo, length, seed=0):
    """Largest error of the estimate over its bound."""
    rng = np.random.default_rng(seed)
    pi = (O.rotation(seed, D)[0] * f32(length)).astype(f32)
    x = rng.standard_normal((48, D)).astype(f32) * np.exp(rng.standard_normal((48, 1))).astype(f32)
    if not lo:
        x = x.astype(f16).astype(f32)
    nrm = np.sqrt((x * x).sum(axis=1, dtype=f32)).astype(f32)[:, None]
    u = (x / nrm).astype(f32)
    y = np.zeros((len(x), D), f32)
    for d in range(D):
        y = (y + (u[:, d:d + 1] * pi[None, :, d]).astype(f32)).astype(f32)
    ph, pl = _pair((pi * f32(256)).astype(f32))
    s = (f32(256) * (f32(1) / nrm)).astype(f32)
    xh, xl = _pair((x * s).astype(f32)) if lo else (x.astype(f64), None)
    acc = np.zeros((len(x), D))
    steps = [slice(c, c + 32) for c in range(0, D, 32)]
    for k in steps:
        acc = _mfma(acc, xh[:, k], pl[:, k])
        if lo:
            acc = _mfma(acc, xl[:, k], ph[:, k])
    for k in steps:
        acc = _mfma(acc, xh[:, k], ph[:, k])
    est = acc / 65536 if lo else acc * ((f32(1) / nrm) / f32(256)).astype(f64)
    N = np.sqrt((pi.astype(f64) ** 2).sum(axis=1))
    return float((np.abs(est - y) / (_bound() * D * 2.0 ** -22 * N)).max())


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("lo", [False, True], ids=["fp16", "fp32"])
def test_estimate_within_its_bound(D, lo):
    assert "!(ss >= 0x1p-16f && ss <= 2500.0f)" in HEADER   # the row lengths that the estimate takes
    for length in (2.0 ** -8, 1.0, 49.0):
        assert _worst(D, lo, length) < 1.0, length
    assert _worst(D, lo, 1e-6) > 1.0
