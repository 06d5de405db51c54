"""Keys of an fp32 pool where the group encode's phases can go wrong, bit for
bit against the oracle (turboquant_pro/per_channel_kv.py:269-401): channels
with large offsets (levels too close for the bucketed codes) beside centred and
constant ones, NaN and infinities, ties at the outlier threshold, more than
eight outliers a channel, groups that are not whole tiles."""

import numpy as np
import pytest

from oracle import tq_oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no ROCm GPU visible")


def _keys(seed, H, L, D):
    rng = np.random.default_rng(seed)
    k = rng.standard_normal((H, L, D)).astype(np.float32)
    k *= np.exp(rng.standard_normal((H, 1, D))).astype(np.float32)
    k[0, :, 1] += 1000.0
    k[0, :, 2] = 1e6 + 1e-2 * k[0, :, 2]          # levels a few ulps apart
    k[0, :, 3] = 0.0
    k[0, :, 4] = 7.25                              # constant: every magnitude tied
    k[0, :, 5] = np.sign(k[0, :, 5]) * 3.0
    k[0, :, 6] *= 1e30
    k[0, :, 7] *= 1e-30
    k[H - 1, 3, 9] = np.nan
    k[H - 1, 4, 10] = np.inf
    k[H - 1, 5, 10] = -np.inf
    return k


@pytest.mark.parametrize("D,W,frac,grid,bits", [
    (128, 512, 0.02, "nf4_asym", 4), (128, 512, 0.1, "nf4_asym", 4), (128, 37, 0.02, "nf4_asym", 4),
    (64, 130, 0.05, "nf4_asym", 4), (256, 512, 0.02, "nf4_asym", 4), (128, 512, 0.02, "uniform", 3),
    (256, 66, 0.0, "uniform", 2), (64, 16, 0.02, "nf4_asym", 4)])
def test_f32_keys_match_oracle(D, W, frac, grid, bits):
    from turboquant_pro_amd import TQKVPool
    print(f"[f32 keys] D={D} W={W} frac={frac} {grid}{bits}", flush=True)
    H, G = 2, (W + 1) // 2
    L = W + 1 + G
    k = _keys(D + W, H, L, D)
    pool = TQKVPool(n_kv_heads=H, head_dim=D, max_batch=1, max_seq_len=L, hot_window=W, key_bits=bits,
                    outlier_frac=frac, key_grid=grid, outlier_cap=G * D if frac else None, seed=0,
                    input_dtype="float32")
    kt = torch.from_numpy(k[None]).cuda()
    pool.append(kt, torch.zeros_like(kt))
    with np.errstate(all="ignore"):
        for g in range(2):
            x = k[:, g * G:(g + 1) * G]
            want = O.encode_keys(x, frac) if grid == "nf4_asym" else O.encode_keys_uniform(x, frac, bits)
            e = pool.export_group(0, g)
            assert np.array_equal(e["kpacked"], want.packed), f"group {g}: codes"
            assert np.array_equal(e["nf4_scale"].view(np.uint32), want.nf4_scale.view(np.uint32))
            assert np.array_equal(e["nf4_mean"].view(np.uint32), want.nf4_mean.view(np.uint32))
            if frac:
                assert np.array_equal(e["outlier_idx"], want.outlier_idx), f"group {g}: outliers"
                assert np.array_equal(e["outlier_val"].view(np.uint16), want.outlier_val.view(np.uint16))
