"""The NF4 codes by bucket, restated in NumPy, against the argmin over all 16
levels (turboquant_pro/per_channel_kv.py:346-383): a bucket of the normalised
key names two neighbouring levels and one comparison with an fp16 threshold
decides.  Every fp16 number of a channel's range is checked, for channels from
centred ones to the largest offsets whose levels count as far enough apart."""

import os
import re

import numpy as np
import pytest

from turboquant_pro_amd.formats import NF4

_SOURCE = open(os.path.join(os.path.dirname(__file__), "..", "turboquant-pro_amd", "csrc", "tqk_encode.hip")).read()
# first bucket of every level pair: the kernels' table
FROM = [int(x) for x in re.search(r"kNf4From\[16\] = \{([^}]*)\}", _SOURCE).group(1).split(",")]
PAIR = np.repeat(np.arange(15), np.diff(FROM))
f32 = np.float32


def _levels(mu, amax):
    return (f32(mu) + f32(amax) * NF4).astype(f32)


def _crowded(mu, amax):
    return not np.all(np.diff(_levels(mu, amax)) >= (abs(f32(mu)) + f32(amax)) * f32(2.0 ** -18))


def _fp16_between(lo, hi):
    x = np.arange(65536, dtype=np.uint16).view(np.float16)
    x = x[np.isfinite(x)].astype(f32)
    return x[(x >= lo) & (x <= hi)]


def _thresholds(c):
    """Smallest fp16 number that the two-level argmin puts on the upper level."""
    x = np.sort(_fp16_between(-65504, 65504))
    out = np.full(15, np.inf, f32)
    for k in range(15):
        up = (x >= c[k + 1]) | ((x > c[k]) & (np.abs(x - c[k + 1]) < np.abs(x - c[k])))
        if up.any():
            assert up[np.argmax(up):].all()  # monotone: the kernel's search relies on it
            out[k] = x[np.argmax(up)]
    return out


def test_table_covers_the_buckets():
    assert len(FROM) == 16 and FROM[0] == 0 and FROM[15] == 32 and np.all(np.diff(FROM) > 0)


def test_every_bucket_holds_at_most_its_own_midpoint():
    mid = (NF4[:-1].astype(np.float64) + NF4[1:]) / 2
    for i in range(32):
        lo, hi = -1 + i / 16 - 0.004, -1 + (i + 1) / 16 + 0.004
        assert not [k for k in range(15) if lo <= mid[k] <= hi and k != PAIR[i]]


@pytest.mark.parametrize("mu,amax", [(0.0, 1.0), (0.0, 1e-8), (0.3, 0.7), (-1.25, 3.5), (17.0, 0.9), (900.0, 25.0),
                                     (-3.0, 40000.0), (250.0, 0.05), (1000.0, 0.06), (-0.0004, 0.0011),
                                     (0.039793, 1.0), (60000.0, 4000.0)])
def test_bucket_codes_equal_argmin(mu, amax):
    if _crowded(mu, amax):
        pytest.skip("levels too close for the buckets: the kernel takes the argmin")
    c = _levels(mu, amax)
    x = _fp16_between(f32(mu) - f32(amax), f32(mu) + f32(amax))
    x = x[np.abs(x - f32(mu)) <= f32(amax)]
    t = (x - f32(mu)) * (f32(15.9995) / f32(amax)) + f32(16)
    i = np.minimum(np.maximum(t, 0).astype(np.int64), 32)
    assert i.max(initial=0) < 32
    k = PAIR[i]
    got = k + (x >= _thresholds(c)[k])
    want = np.argmin(np.abs(x[:, None] - c), axis=1)
    assert np.array_equal(got, want)
