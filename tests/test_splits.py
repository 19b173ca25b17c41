"""The decode attention's split count (host rule, no GPU)."""
import pytest

from litemoe_amd.flash_decode import default_splits


@pytest.mark.parametrize("batch,kv_heads,maximum,splits", [
    (1, 8, 512, 1), (1, 8, 767, 1), (1, 8, 768, 3), (1, 8, 4096, 16), (3, 8, 4001, 10), (10, 8, 2000, 3),
    (32, 8, 4096, 1), (33, 8, 4096, 2), (64, 8, 4096, 1), (128, 8, 4096, 1), (0, 8, 4096, 16), (1, 1, 16, 1)])
def test_default_splits(batch, kv_heads, maximum, splits):
    assert default_splits(batch, kv_heads, maximum) == splits


def test_default_splits_keep_min_keys_and_the_cap():
    for maximum in range(1, 5000, 37):
        for batch in (1, 2, 5, 17, 40, 200):
            n = default_splits(batch, 8, maximum)
            assert 1 <= n <= 16 and (n == 1 or maximum // n >= 256)


@pytest.mark.parametrize("batch,maximum,splits", [
    (16, 4096, 2), (17, 3071, 1), (17, 3072, 3), (17, 4096, 3), (19, 4096, 3), (20, 4096, 1)])
def test_default_splits_of_long_contexts_do_not_leave_half_the_cus_idle(batch, maximum, splits):
    """At 17 to 19 rows of 8 heads one workgroup per pair leaves 104 to 120 of the
    256 CUs without one; three splits fill them where the keys suffice."""
    assert default_splits(batch, 8, maximum) == splits
