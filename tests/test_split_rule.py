"""Split counts of the fused decode where the row groups do not divide the CUs
(256 without a device): no nearly empty last round of workgroups."""

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
