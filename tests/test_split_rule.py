"""Split counts of the decode kernels (256 CUs without a device): of the fused one
where the row groups do not divide the CUs, no nearly empty last round of
workgroups; of many query rows, what the three-call form can run."""

import pytest

from quashkv_amd import _native as N


@pytest.mark.parametrize("B,Hq,Hkv,d,T,splits", [
    (12, 24, 8, 96, 3001, 2),     # 96 groups: 3 splits would be 288 workgroups
    (12, 32, 8, 128, 3001, 2),
    (20, 32, 8, 128, 2000, 1),    # 160 groups
    (5, 56, 8, 128, 6000, 3),     # 80 groups (7 rows in two chunks): 240 workgroups
    (8, 32, 8, 128, 65536, 4),    # 64 groups: a divisor, as before
    (32, 32, 8, 128, 65536, 1),
])
def test_splits_of_odd_group_counts(B, Hq, Hkv, d, T, splits):
    assert N.lib().qkv_attention_splits(B, Hq, Hkv, 1, d, T) == splits


@pytest.mark.parametrize("B,Hq,Hkv,Q,d,T,splits", [
    (8, 32, 8, 64, 64, 8192, 4),      # split_mfma's scores fit LDS up to 2048 tokens a split
    (1, 8, 8, 48, 64, 65536, 32),
    (1, 8, 8, 256, 128, 2048, 1),     # 512 row groups: no splits, whatever the prefill kernel likes
    (2, 8, 4, 64, 96, 4096, 1),
])
def test_splits_of_many_rows_serve_the_three_call_form(B, Hq, Hkv, Q, d, T, splits):
    L = N.lib()
    s = L.qkv_attention_splits(B, Hq, Hkv, Q, d, T)
    assert s == splits
    if d == 64:
        assert -(-T // s) <= 2048
    # room for the decode layout, and for the prefill kernel's splits
    R = Hq // Hkv * Q
    rows, ch = B * Hkv * R, B * Hkv * ((R + 3) // 4)
    layout = rows * 8 * d + ch * (6 * 64 * 16 + 32) + s * rows * (4 * d + 8)
    own = min(64, 256 // (B * Hkv * ((R + 127) // 128)))
    room = max(1, own) * rows * (4 * d + 8)
    assert L.qkv_attention_workspace_bytes(B, Hq, Hkv, Q, d, s) == max(layout, room)


@pytest.mark.parametrize("B,H,R,T,kb,ranges,prefills", [
    # decode_small serves the call: 21 us against 26
    (20, 5, 287, 95, 3, 0, False), (20, 5, 287, 500, 3, 0, True), (1, 8, 48, 256, 3, 0, False),
    # it does not (3 key MSE bits; key ranges): 330 and 290 us
    (20, 5, 287, 95, 4, 0, True), (20, 5, 287, 95, 3, 1, True), (4, 8, 64, 400, 4, 0, True),
    (1, 8, 48, 256, 4, 0, False), (1, 8, 47, 4096, 4, 0, False),
])
def test_prefill_rule_at_64(B, H, R, T, kb, ranges, prefills):
    L = N.lib()
    m = [0.05, 0.15, 0.25, 0.35][: 1 << (kb - 2)]
    kc = N.HostFloats([-x for x in m[::-1]] + m)
    vc = N.HostFloats([-2.0, -1.3, -0.7, -0.2, 0.2, 0.7, 1.3, 2.0])
    s = L.qkv_attention_splits(B, H, H, R, 64, T)
    ws = L.qkv_attention_workspace_bytes(B, H, H, R, 64, s)
    n = L.qkv_attention_prefills(B, H, H, R, 64, T, kb - 1, 3, kc.ptr, vc.ptr, 0.02,
                                 -(-T // 64) * 64, ranges, ws, s)
    assert (n > 0) == prefills
