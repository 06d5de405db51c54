"""The key-block encode over its routes: ``tqk_key_block_stats`` and what follows
it over the chip, and ``tqk_key_block``, one workgroup per (batch, head), for
blocks with outliers too small for what the former hand on through the packed
output.  Both find the threshold of turboquant_pro/per_channel_kv.py:274-280
(np.partition's k-th largest magnitude, every magnitude at or above it an
entry).

``test_threshold_paths_agree``: a side-list capacity below head_dim gives the
same codes, scale, zero point and count as a large one, its entries being the
first ones of the large one's: fp16 and fp32 input, asym-NF4 and uniform 4-bit
keys, lognormal channel scales, magnitude ties at the threshold and a NaN.
``test_routes_match_oracle``: both routes against the oracle on either side of
the rule between them, at the edges of the 256-token chunks and 512-token
tiles, with every element an outlier, with small capacities, and with input and
packed output at addresses that are multiples of one element and one byte.
"""

import ctypes

import numpy as np
import pytest

from oracle import tq_oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no ROCm GPU visible")


def _encode(x, uniform, k, cap):
    from turboquant_pro_amd import _native as N
    from turboquant_pro_amd.plugins import _block_desc
    B, H, S, D = x.shape
    dev = x.device
    kp = torch.zeros(B * H * S * D // 2, dtype=torch.uint8, device=dev)
    scale = torch.zeros((B, H, D), dtype=torch.float32, device=dev)
    zero = torch.zeros_like(scale)
    count = torch.zeros(B * H, dtype=torch.int32, device=dev)
    pos = torch.zeros((B * H, cap), dtype=torch.int32, device=dev)
    val = torch.zeros((B * H, cap), dtype=torch.float16, device=dev)
    d = _block_desc(x.shape, 4, int(uniform), 0, k, cap, int(x.dtype == torch.float32), None)
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    N.check(N.lib().tqk_encode_key_block(ctypes.byref(d), x.data_ptr(), None, kp.data_ptr(),
                                         scale.data_ptr(), zero.data_ptr(), pos.data_ptr(),
                                         val.data_ptr(), count.data_ptr(), st), "tqk_encode_key_block")
    torch.cuda.synchronize()
    return [t.cpu().numpy() for t in (kp, scale, zero, count, pos, val)]


@pytest.mark.parametrize("dtype", ["float16", "float32"])
@pytest.mark.parametrize("uniform", [False, True], ids=["nf4_asym", "uniform4"])
@pytest.mark.parametrize("S", [300, 1000])
def test_threshold_paths_agree(dtype, uniform, S):
    from turboquant_pro_amd.codebooks import outliers_per_channel
    B, H, D = 1, 2, 128
    print(f"[key-block] threshold paths dtype={dtype} uniform={uniform} S={S}", flush=True)
    rng = np.random.default_rng(S + 7 * uniform)
    x = rng.standard_normal((B, H, S, D)).astype(np.float32)
    x *= np.exp(0.7 * rng.standard_normal((1, H, 1, D))).astype(np.float32)
    x[0, 0, :, 5] = 0.1 * rng.standard_normal(S)
    x[0, 0, : S // 4, 5] = 3.0          # the channel's largest magnitude, S / 2 times,
    x[0, 0, S // 4: S // 2, 5] = -3.0   # of both signs: ties at its threshold
    x[0, 1, 17, 9] = np.nan             # a NaN orders above every magnitude
    xt = torch.from_numpy(x).to(getattr(torch, dtype)).cuda()
    k = outliers_per_channel(S, 0.02)
    big = _encode(xt, uniform, k, 4 * k * D)
    small = _encode(xt, uniform, k, D // 2)
    for name, a, b in zip(("codes", "scale", "zero", "count"), big[:4], small[:4]):
        assert np.array_equal(a.view(np.uint8), b.view(np.uint8)), name
    cnt = big[3]
    assert cnt[0] >= (D - 1) * k + S // 2   # the ties keep every equal magnitude
    for i in range(B * H):
        n = min(int(cnt[i]), D // 2)
        assert np.array_equal(big[4][i, :n], small[4][i, :n]), f"positions of (b, h) {i}"
        assert np.array_equal(big[5][i, :n].view(np.uint16), small[5][i, :n].view(np.uint16)), \
            f"values of (b, h) {i}"


@pytest.mark.parametrize("D,bits,grid,S,frac,dtype,cap,x_off,p_off", [
    # the rule: D + chunks + S D / 32 dwords in S D bits / 32 of them
    (128, 2, "uniform", 32, 0.05, "float32", 0, 0, 0), (128, 2, "uniform", 33, 0.05, "float32", 0, 0, 0),
    (128, 2, "uniform", 33, 0.05, "float16", 0, 1, 3), (64, 3, "uniform", 16, 0.1, "float16", 0, 0, 0),
    (64, 3, "uniform", 17, 0.1, "float16", 0, 0, 0), (64, 3, "uniform", 18, 0.1, "float32", 0, 1, 1),
    (256, 4, "nf4", 10, 0.1, "float32", 0, 0, 0), (256, 4, "nf4", 11, 0.1, "float32", 0, 0, 0),
    (256, 4, "nf4", 11, 0.1, "float16", 0, 0, 2), (128, 4, "nf4", 1, 0.02, "float16", 0, 0, 0),
    # chunks and tiles
    (64, 4, "nf4", 256, 0.02, "float16", 0, 0, 0), (64, 4, "uniform", 257, 0.02, "float32", 0, 0, 0),
    (128, 4, "nf4", 512, 0.02, "float32", 0, 0, 0), (128, 3, "uniform", 513, 0.02, "float16", 0, 0, 0),
    (256, 4, "nf4", 513, 0.02, "float16", 0, 0, 0), (256, 2, "uniform", 512, 0.02, "float32", 0, 0, 0),
    # up to 128 tokens the threshold by counting, up to 128 of a chunk codes by pieces
    (128, 2, "uniform", 64, 0.1, "float32", 0, 0, 0), (64, 3, "uniform", 65, 0.1, "float16", 0, 0, 0),
    (256, 3, "uniform", 128, 0.2, "float32", 0, 0, 1), (64, 2, "uniform", 129, 0.1, "float32", 0, 0, 0),
    (128, 3, "uniform", 384, 0.02, "float16", 0, 1, 3), (256, 2, "uniform", 385, 0.02, "float32", 0, 0, 0),
    # every element an outlier, and none
    (128, 4, "nf4", 9, 1.0, "float32", 0, 0, 0), (64, 4, "nf4", 300, 1.0, "float16", 0, 0, 0),
    (128, 4, "nf4", 300, 0.0, "float32", 0, 1, 1), (256, 2, "uniform", 40, 0.0, "float16", 0, 1, 2),
    # small capacities, odd addresses
    (128, 4, "nf4", 700, 0.02, "float32", 5, 0, 0), (256, 4, "uniform", 300, 0.02, "float16", 100, 0, 0),
    (128, 4, "nf4", 700, 0.02, "float32", 0, 1, 0), (64, 4, "nf4", 700, 0.02, "float16", 0, 3, 1),
    (256, 4, "uniform", 300, 0.02, "float16", 0, 1, 0), (128, 4, "nf4", 300, 0.02, "float32", 0, 0, 2)])
def test_routes_match_oracle(D, bits, grid, S, frac, dtype, cap, x_off, p_off):
    from turboquant_pro_amd import _native as N
    from turboquant_pro_amd.plugins import _block_desc
    print(f"[key-block] routes D={D} bits={bits} {grid} S={S} frac={frac} {dtype} cap={cap} "
          f"off={x_off},{p_off}", flush=True)
    B, H, uniform = 1, 3, grid == "uniform"
    rng = np.random.default_rng(S + D + bits)
    x = rng.standard_normal((H, S, D)).astype(np.float32)
    x *= np.exp(0.7 * rng.standard_normal((H, 1, D))).astype(np.float32)
    x[0, :, 5] = np.float32(0.5) * np.sign(x[0, :, 5])   # ties, of both signs
    x[1, :, 7] = 0.0
    x = x.astype(dtype).astype(np.float32)
    k = O.outlier_count_per_channel(S, frac) if frac else 0
    want = O.encode_keys_uniform(x, frac, bits) if uniform else O.encode_keys(x, frac)
    cap = cap or max(S * D, 1)
    n = H * S * D
    xt = torch.zeros(n + 8, dtype=getattr(torch, dtype), device="cuda")
    xt[x_off:x_off + n] = torch.from_numpy(x.reshape(-1)).cuda().to(xt.dtype)
    nb = n * bits // 8
    kp = torch.full((nb + 16,), 0xA5, dtype=torch.uint8, device="cuda")
    scale = torch.zeros((H, D), dtype=torch.float32, device="cuda")
    zero = torch.zeros_like(scale)
    count = torch.full((H,), -1, dtype=torch.int32, device="cuda")
    pos = torch.full((H + 1, cap), -1, dtype=torch.int32, device="cuda")
    val = torch.zeros((H + 1, cap), dtype=torch.float16, device="cuda")
    d = _block_desc((B, H, S, D), bits, int(uniform), 0, k, cap, int(dtype == "float32"), None)
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    N.check(N.lib().tqk_encode_key_block(
        ctypes.byref(d), xt.data_ptr() + x_off * xt.element_size(), None, kp.data_ptr() + p_off, scale.data_ptr(),
        zero.data_ptr(), pos.data_ptr(), val.data_ptr(), count.data_ptr(), st), "tqk_encode_key_block")
    torch.cuda.synchronize()
    got = kp.cpu().numpy()
    assert np.array_equal(got[p_off:p_off + nb], want.packed)
    assert np.all(got[:p_off] == 0xA5) and np.all(got[p_off + nb:] == 0xA5)
    assert np.array_equal(scale.cpu().numpy(), want.nf4_scale)
    assert np.array_equal(zero.cpu().numpy(), want.nf4_mean)
    assert np.all(pos[H].cpu().numpy() == -1)
    idx = np.zeros(0, np.int64) if want.outlier_idx is None else want.outlier_idx.astype(np.int64)
    for h in range(H):
        m = idx // (S * D) == h
        assert int(count[h]) == int(m.sum())
        e = min(int(m.sum()), cap)
        assert np.array_equal(pos[h, :e].cpu().numpy(), (idx[m] - h * S * D)[:e])
        assert np.all(pos[h, e:].cpu().numpy() == -1)
        if e:
            assert np.array_equal(val[h, :e].cpu().numpy().view(np.uint16), want.outlier_val[m][:e].view(np.uint16))


@pytest.mark.parametrize("D,frac", [(256, 0.0), (64, 0.3)])
def test_more_heads_than_a_launch_takes(D, frac):
    """262147 heads of head_dim 256 (and 1048579 of 64, with a side-list) would be more than
    2^32 threads in one launch; the first and last of them and those around the cuts as in
    blocks of their own."""
    from turboquant_pro_amd import _native as N
    from turboquant_pro_amd.plugins import _block_desc
    cut, S = (1 << 21) // (D // 16), 1 if frac == 0.0 else 13
    H, k = 2 * cut + 3, int(round(S * frac))
    print(f"[key-block] {H} heads of {S} x {D}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(D)
    x = torch.randn((H, S, D), generator=gen, device="cuda", dtype=torch.float16)

    def encode(x):
        n, cap = x.shape[0], 2 * D * max(k, 1)
        kp = torch.zeros((n, S * D // 2), dtype=torch.uint8, device="cuda")
        scale = torch.zeros((n, D), dtype=torch.float32, device="cuda")
        zero = torch.zeros_like(scale)
        count = torch.full((n,), -1, dtype=torch.int32, device="cuda")
        pos = torch.zeros((n, cap), dtype=torch.int32, device="cuda")
        val = torch.zeros((n, cap), dtype=torch.float16, device="cuda")
        d = _block_desc((1, n, S, D), 4, 0, 0, k, cap, 0, None)
        st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        N.check(N.lib().tqk_encode_key_block(
            ctypes.byref(d), x.data_ptr(), None, kp.data_ptr(), scale.data_ptr(), zero.data_ptr(), pos.data_ptr(),
            val.data_ptr(), count.data_ptr(), st), "tqk_encode_key_block")
        return kp, scale, zero, count, pos, val

    whole = encode(x)
    for a, b in ((0, 2), (cut - 2, cut + 2), (2 * cut - 2, 2 * cut + 3)):
        for got, want in zip(whole, encode(x[a:b].contiguous())):
            assert torch.equal(got[a:b], want)
    assert int(whole[3].min()) >= D * k
