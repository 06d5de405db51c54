"""The decode of fp32 caches at their side-list: entries whose dense part is a
code of the row (2-, 3- and 4-bit keys), lists that fit the 2048 entries staged
in LDS and lists that do not, 1 to 8 query heads, against the oracle."""

import numpy as np
import pytest

from gpu_util import assert_attn_close
from oracle import tq_oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no ROCm GPU visible")


# side-list entries of a group: ceil(frac * G) * D
@pytest.mark.parametrize("D,Hq,W,frac,grid,bits,vb", [
    (64, 1, 512, 0.02, "uniform", 2, 3), (64, 4, 512, 0.125, "uniform", 3, 3),    # 384, 2048: the last to fit
    (64, 4, 512, 0.128, "nf4_asym", 4, 3), (128, 2, 512, 0.02, "uniform", 3, 3),  # 2112: the first not to; 768
    (128, 7, 37, 0.1, "uniform", 2, 3), (128, 4, 512, 0.1, "nf4_asym", 4, 3),     # 256; 3328
    (256, 2, 512, 0.02, "uniform", 2, 3), (256, 8, 66, 0.05, "nf4_asym", 4, 3),
    # codes and rows in other arrays' places: rows only, and both
    (256, 1, 512, 0.02, "nf4_asym", 4, 4), (256, 1, 37, 0.3, "uniform", 3, 4),
    (64, 4, 512, 0.02, "nf4_asym", 4, 2), (64, 3, 37, 0.3, "uniform", 2, 2)])
def test_decode_matches_oracle(D, Hq, W, frac, grid, bits, vb):
    """Tolerance: the oracle test's own bar for fp32 caches (2e-4); one wrong
    code moves a score by at least a level's step of its channel."""
    from turboquant_pro_amd import TQKVPool
    print(f"[f32 side-list] D={D} Hq={Hq} W={W} frac={frac} {grid}{bits} V{vb}", flush=True)
    G = (W + 1) // 2
    L = W + 1 + 2 * G + 3
    k, v, q = (x.astype(np.float32) for x in O.synthetic_kv(D + W + Hq, 1, 1, Hq, L, D=D))
    k *= np.float32(1.0009765625 / 3)    # off the fp16 grid
    pi, pi_t = O.rotation(3, D)
    sc = O.SequenceCache(hot_window=W, value_bits=vb, outlier_frac=frac, key_grid=grid, key_bits=bits).build(
        k[0], v[0], pi, pi_t)
    pool = TQKVPool(n_kv_heads=1, n_q_heads=Hq, head_dim=D, max_batch=1, max_seq_len=L, hot_window=W,
                    value_bits=vb, key_bits=bits, key_grid=grid, outlier_frac=frac, outlier_cap=G * D,
                    rotation=(pi, pi_t), input_dtype="float32")
    pool.append(*(torch.from_numpy(x).cuda() for x in (k, v)))
    got = pool.decode(torch.from_numpy(q).cuda()).cpu().numpy()
    assert_attn_close(got[0], sc.attend(q[0]), atol=2e-4, rtol=1e-3, what=f"D={D} frac={frac} {grid}{bits}")
