"""The VALU decode's split plan, read from the workspace size: never more splits
than the model's three workgroups a CU give, and fewer only where it counts four."""

import ctypes

import pytest

from test_abi_cpu import _desc, _lib

CUS = 256  # the plan's count without a device


def _three(pairs, groups, hot):
    """Groups per split that cost least with three workgroups a CU."""
    units = pairs * groups
    lo = -(-units // 4096) if units > 4096 else 1
    hi = max(lo, min(8 * lo, groups))
    return min(range(lo, hi + 1), key=lambda g: (-(-pairs * (-(-groups // g) + hot) // (3 * CUS)) * (g + 1), g))


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("gq", [1, 2, 4, 7])
@pytest.mark.parametrize("vb", [2, 3, 4])
def test_splits(D, gq, vb):
    import torch
    if torch.cuda.is_available():
        pytest.skip("restates the plan for the CU count used without a device")
    N, lib = _lib()
    hkv, hot = 2, 2
    d = _desc(N, n_kv_heads=hkv, n_q_heads=hkv * gq, head_dim=D, value_bits=vb, input_f32=1,
              max_groups_per_seq=400, max_pages_per_seq=400 * 16)
    four = D <= 128 and gq <= 4 and not (vb == 4 and D == 128 and gq == 4)
    fewer = 0
    for batch in (1, 3, 16, 32, 64):
        def partials(length):
            return lib.tqk_decode_workspace_bytes(ctypes.byref(d), batch, length) - 256

        per = batch * hkv * gq * 4 * (2 + D)  # bytes of one split
        fixed = partials(1) - per             # counters
        for groups in (1, 2, 7, 30, 63, 200, 399):
            splits = (partials(512 + 256 * (groups - 1) + 1) - fixed) // per - hot
            want = -(-groups // _three(batch * hkv, groups, hot))
            assert splits == want or (four and splits < want), (batch, groups, splits, want)
            fewer += splits < want
    assert (fewer > 0) == four
