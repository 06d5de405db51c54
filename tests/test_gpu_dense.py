"""Dense keys and values of a pool in one call (``TQKVPool.dense``), bit for bit
against the oracle's reconstruction (turboquant_pro/per_channel_kv.py:497-539,
turboquant_pro/core.py:619-654) rounded to the output type, ragged lengths and
groups that are not whole 64-token chunks among them."""

import numpy as np
import pytest

from oracle import tq_oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no ROCm GPU visible")


@pytest.mark.parametrize("D,W,vb,lens,dtype,out", [
    (128, 512, 3, (1300, 40), "float16", "bfloat16"), (128, 512, 4, (769, 768), "float16", "float16"),
    (128, 48, 2, (200, 49), "float16", "float32"), (64, 130, 3, (500, 1), "float16", "bfloat16"),
    (256, 66, 4, (140, 67), "float16", "float16"), (128, 512, 3, (1025, 513), "float32", "bfloat16")])
def test_dense_matches_oracle(D, W, vb, lens, dtype, out):
    from turboquant_pro_amd import TQKVPool
    print(f"[dense] D={D} W={W} V{vb} {lens} {dtype} -> {out}", flush=True)
    H, L = 2, max(lens)
    k, v, _ = O.synthetic_kv(D + W + vb, 2, H, H, L, D=D)
    pool = TQKVPool(n_kv_heads=H, head_dim=D, max_batch=2, max_seq_len=L, hot_window=W, value_bits=vb, seed=0,
                    input_dtype=dtype)
    kt, vt = (torch.from_numpy(x).cuda().to(pool.dtype) for x in (k, v))
    pool.append(kt, vt, n_new=list(lens))
    gk, gv = pool.dense(getattr(torch, out))
    pi, pi_t = O.rotation(0, D)
    for b, n in enumerate(lens):
        x = kt.cpu().numpy() if dtype == "float32" else k
        y = vt.cpu().numpy() if dtype == "float32" else v
        seq = O.SequenceCache(hot_window=W, value_bits=vb, outlier_frac=0.02).build(
            x[b][:, :n], y[b][:, :n], pi, pi_t)
        for got, want in ((gk, seq.get_keys()), (gv, seq.get_values())):
            want = torch.from_numpy(np.asarray(want, np.float32).reshape(H, n, D)).to(getattr(torch, out))
            assert torch.equal(got[b, :, :n].cpu(), want)
