"""The group encode's instances (by the largest group they take: 64, 128 and 256
tokens) at the edges of the rule between them, bit for bit against the oracle
(turboquant_pro/per_channel_kv.py:269-401, core.py:542-617): keys, side-list,
value codes and norms of two groups."""

import numpy as np
import pytest

from oracle import tq_oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no ROCm GPU visible")


@pytest.mark.parametrize("dtype", ["float16", "float32"])
@pytest.mark.parametrize("D,G,vb,frac,grid,bits", [
    (64, 1, 3, 0.0, "uniform", 2), (64, 64, 3, 0.02, "nf4_asym", 4), (64, 65, 3, 0.02, "nf4_asym", 4),
    (64, 128, 4, 0.05, "uniform", 3), (64, 129, 2, 0.02, "nf4_asym", 4), (128, 64, 3, 0.2, "nf4_asym", 4),
    (128, 64, 4, 0.02, "uniform", 4), (128, 65, 3, 0.02, "nf4_asym", 4), (128, 8, 2, 0.2, "nf4_asym", 4),
    (256, 64, 3, 0.02, "nf4_asym", 4), (256, 64, 2, 0.15, "uniform", 2), (256, 65, 4, 0.02, "nf4_asym", 4),
    (256, 33, 4, 0.0, "nf4_asym", 4)])
def test_groups_match_oracle(D, G, vb, frac, grid, bits, dtype):
    from turboquant_pro_amd import TQKVPool
    print(f"[encode groups] D={D} G={G} V{vb} frac={frac} {grid}{bits} {dtype}", flush=True)
    H, W = 3, 2 * G
    L = W + 1 + G
    rng = np.random.default_rng(D + G)
    k, v = (rng.standard_normal((H, L, D)).astype(np.float32) for _ in range(2))
    k *= np.exp(0.7 * rng.standard_normal((H, 1, D))).astype(np.float32)
    k[0, :, 3] += 200.0
    v[1, ::5] = 0.0
    k, v = k.astype(dtype), v.astype(dtype)
    pi, pi_t = O.rotation(3, D)
    _, bnd = O.polar_codebook(vb, D)
    pool = TQKVPool(n_kv_heads=H, head_dim=D, max_batch=1, max_seq_len=L, hot_window=W, value_bits=vb, key_bits=bits,
                    key_grid=grid, outlier_frac=frac, outlier_cap=G * D if frac else None, rotation=(pi, pi_t),
                    input_dtype=dtype)
    pool.append(torch.from_numpy(k[None]).cuda(), torch.from_numpy(v[None]).cuda())
    for g in range(2):
        x = k[:, g * G:(g + 1) * G].astype(np.float32)
        want = O.encode_keys(x, frac) if grid == "nf4_asym" else O.encode_keys_uniform(x, frac, bits)
        val = O.encode_values(v[:, g * G:(g + 1) * G].astype(np.float32), pi_t, bnd, vb)
        e = pool.export_group(0, g)
        assert np.array_equal(e["kpacked"], want.packed), f"group {g}: key codes"
        assert np.array_equal(e["nf4_scale"], want.nf4_scale) and np.array_equal(e["nf4_mean"], want.nf4_mean)
        if frac:
            assert np.array_equal(e["outlier_idx"], want.outlier_idx), f"group {g}: outliers"
            assert np.array_equal(e["outlier_val"].view(np.uint16), want.outlier_val.view(np.uint16))
        assert np.array_equal(e["vpacked"], val.packed), f"group {g}: value codes"
        assert np.array_equal(e["vnorms"], val.norms), f"group {g}: norms"
