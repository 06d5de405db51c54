"""PolarQuant codes where the matrix-core estimate may not decide them, bit for
bit against the oracle's ordered sums (turboquant_pro/core.py:542-617): rows
of zeros, of fp16 subnormals, of magnitudes whose squares vanish or overflow,
of NaN, and rotations that put whole channels on a code boundary (identity on
one-hot rows: more flagged codes than the list holds) or lie outside the
estimate's bound (rows of length 100; rows of length 1e-6, whose fp16 halves
are subnormal)."""

import numpy as np
import pytest

from oracle import tq_oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no ROCm GPU visible")


def _rotation(name, D):
    if name == "identity":
        return np.eye(D, dtype=np.float32), np.eye(D, dtype=np.float32)
    pi, pi_t = O.rotation(3, D)
    f = np.float32({"long": 100.0, "short": 1e-6}.get(name, 1.0))
    return np.ascontiguousarray(pi * f), np.ascontiguousarray(pi_t * f)


def _rows(seed, H, L, D, f32):
    """Value rows with the special ones spread over tiles and batches."""
    rng = np.random.default_rng(seed)
    v = rng.standard_normal((H, L, D)).astype(np.float32)
    v[:, 3::16] *= 1e-30 if f32 else 1e-6          # squares that vanish; fp16 subnormals
    v[:, 7::32] = 0.0
    v[:, 8::64] = -0.0
    v[0, 9::64] = 0.0
    v[0, 9::64, 5 % D] = 2.0                          # one-hot
    if f32:
        v[:, 20] *= 1e25                              # the sum of squares overflows
        v[:, 21] *= 1e-18
    else:
        v[:, 20] *= 500.0
    v[H - 1, 11, 4] = np.nan
    return v if f32 else v.astype(np.float16)


@pytest.mark.parametrize("D,vb,W,dtype,rot", [
    (128, 3, 512, "float16", "random"), (128, 3, 512, "float16", "identity"), (128, 2, 64, "float16", "long"),
    (128, 4, 130, "float16", "random"), (64, 3, 512, "float16", "random"), (256, 4, 512, "float16", "identity"),
    (256, 2, 37, "float16", "random"), (128, 3, 512, "float32", "random"), (64, 4, 64, "float32", "identity"),
    (256, 3, 300, "float32", "random"), (128, 2, 33, "float32", "long"),
    (128, 3, 512, "float16", "short"), (64, 3, 512, "float32", "short")])
def test_pool_codes_match_oracle(D, vb, W, dtype, rot):
    from turboquant_pro_amd import TQKVPool
    print(f"[polar codes] D={D} V{vb} W={W} {dtype} {rot}", flush=True)
    H, G = 2, (W + 1) // 2
    L = W + 1 + G                                     # two coded groups
    f32 = dtype == "float32"
    v = _rows(D + vb + W, H, L, D, f32)
    k = np.zeros_like(v)
    pi, pi_t = _rotation(rot, D)
    pool = TQKVPool(n_kv_heads=H, head_dim=D, max_batch=1, max_seq_len=L, hot_window=W,
                    value_bits=vb, outlier_frac=0.0, rotation=(pi, pi_t), input_dtype=dtype)
    pool.append(torch.from_numpy(k[None]).cuda(), torch.from_numpy(v[None]).cuda())
    _, bnd = O.polar_codebook(vb, D)
    with np.errstate(all="ignore"):
        for g in range(2):
            want = O.encode_values(v[:, g * G:(g + 1) * G], pi_t, bnd, vb)
            e = pool.export_group(0, g)
            assert np.array_equal(e["vpacked"], want.packed), f"group {g}: codes"
            assert np.array_equal(e["vnorms"].view(np.uint32), want.norms.view(np.uint32)), f"group {g}: norms"


@pytest.mark.parametrize("D,bits,S,dtype", [(128, 3, 1, "float32"), (128, 4, 63, "float16"), (128, 2, 65, "float32"),
                                            (64, 3, 130, "float16"), (256, 4, 70, "float32")])
def test_block_codes_match_oracle(D, bits, S, dtype):
    from turboquant_pro_amd import plugins
    H = 3
    x = _rows(S, H, max(S, 33), D, dtype == "float32")[:, :S]
    q = plugins.create("polar", head_dim=D, n_heads=H, bits=bits, seed=3)
    got = q.compress(x[None], packed=True)
    _, bnd = O.polar_codebook(bits, D)
    with np.errstate(all="ignore"):
        want = O.encode_values(x, q.rotation[1], bnd, bits)
    assert np.array_equal(got.indices, want.packed)
    assert np.array_equal(got.norms[0].view(np.uint32), want.norms.view(np.uint32))
