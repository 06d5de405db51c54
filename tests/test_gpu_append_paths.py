"""An append whose lengths and groups go with the launches (at most 64 sequences
and 128 completed groups) leaves the same cache as one that copies them to the
device: every buffer and length, at the limits and one beyond, one token at a
time and ragged (turboquant_pro/core.py:986-1038)."""

import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no ROCm GPU visible")


def _ragged(B, T):
    return [(b * 7) % (T + 1) for b in range(B)]


@pytest.mark.parametrize("B,W,dtype,appends", [
    (1, 16, "float16", [(1, None)] * 26),                       # a token at a time over a flush
    (3, 16, "float32", [(40, [40, 0, 17]), (1, [0, 1, 1]), (9, [9, 8, 0])]),
    (64, 16, "float16", [(33, None), (5, _ragged(64, 5))]),     # 64 sequences, 3 groups each: beyond 128
    (64, 16, "float16", [(25, None), (5, _ragged(64, 5))]),     # 64 x 2 groups: at 128
    (65, 16, "float16", [(12, _ragged(65, 12))]),               # a sequence too many
    (1, 16, "float16", [(16 + 8 * 127 + 1, None), (7, None), (8 * 129, None)])])
def test_same_cache(B, W, dtype, appends, monkeypatch):
    from turboquant_pro_amd import TQKVPool, _native as N
    print(f"[append paths] B={B} W={W} {dtype}", flush=True)
    H, D = 2, 64
    total = sum(t for t, _ in appends)
    pools = [TQKVPool(n_kv_heads=H, head_dim=D, max_batch=B, max_seq_len=total, hot_window=W, seed=0,
                      input_dtype=dtype) for _ in range(2)]
    gen = torch.Generator(device="cuda").manual_seed(B + total)
    for T, n_new in appends:
        k, v = (torch.randn((B, H, T, D), generator=gen, device="cuda").to(pools[0].dtype) for _ in range(2))
        pools[0].append(k, v, n_new)
        with monkeypatch.context() as m:
            m.setattr(N, "APPEND_SEQS", 0)
            pools[1].append(k, v, n_new)
        assert pools[0].lengths == pools[1].lengths == pools[0].seq_lens.tolist()
        for name in ("seq_lens", "kcodes", "vcodes", "vnorm", "gscale", "gmean", "ocount", "hot_k", "hot_v"):
            a, b = getattr(pools[0], name), getattr(pools[1], name)
            assert torch.equal(a, b), name
        for b in range(0, B, 21):
            for g in range(pools[0].n_groups(b)):
                x, y = pools[0].export_group(b, g), pools[1].export_group(b, g)
                assert all((x[n] == y[n]).all() for n in ("outlier_idx", "outlier_val")), (b, g)


def test_beyond_limits_refused():
    """Nothing is launched past the limits or for a length out of range."""
    import ctypes
    from turboquant_pro_amd import TQKVPool, _native as N
    pool = TQKVPool(n_kv_heads=1, head_dim=64, max_batch=1, max_seq_len=2000, hot_window=16, seed=0)
    T = 16 + 8 * 128 + 1    # 129 groups
    k = torch.zeros((1, 1, T, 64), dtype=torch.float16, device="cuda")
    one = ctypes.c_int32 * 1
    for prev, n, batch in ((0, T, 1), (0, T + 1, 1), (-1, 1, 1), (0, -1, 1), (0, 1, 0)):
        rc = N.lib().tqk_append_tokens(ctypes.byref(pool.desc), ctypes.byref(pool.ptrs), batch, one(prev), one(n),
                                       k.data_ptr(), k.data_ptr(), T, pool.seq_lens.data_ptr(), None, pool._stream())
        assert rc == N.TQK_EINVAL, (prev, n, batch)
    assert pool.seq_lens.tolist() == [0]


def test_more_groups_than_a_launch_takes():
    """65537 one-token groups of 64 heads would be more than 2^32 threads in one
    launch: the same cache as in three appends."""
    from turboquant_pro_amd import TQKVPool
    H, D, L = 64, 64, 65538
    print(f"[append paths] {L - 1} groups of {H} heads", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(5)
    k, v = (torch.randn((1, H, L, D), generator=gen, device="cuda", dtype=torch.float16) for _ in range(2))
    pools = [TQKVPool(n_kv_heads=H, head_dim=D, max_batch=1, max_seq_len=L, hot_window=1, seed=0, outlier_frac=0.0)
             for _ in range(2)]
    pools[0].append(k, v)
    for a, b in ((0, 30000), (30000, 60000), (60000, L)):
        pools[1].append(k[:, :, a:b], v[:, :, a:b])
    for name in ("seq_lens", "kcodes", "vcodes", "vnorm", "gscale", "gmean", "ocount", "hot_k", "hot_v"):
        assert torch.equal(getattr(pools[0], name), getattr(pools[1], name)), name
    assert int(torch.count_nonzero(pools[0].vnorm)) == H * (L - 1)
