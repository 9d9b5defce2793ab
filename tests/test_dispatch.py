"""Which form the attention entry points choose by size (no GPU call is made)."""

import pytest


@pytest.mark.parametrize("HD", [64, 128])
def test_kept_scores_rule(HD):
    """Kept scores only where the other forms would read K twice, with three splits a tile or more and scratch within
    its limit; elsewhere the split of the exchange, one-block and K-twice forms."""
    from bitexact.vllm_plugin.tri_exact_attn import SCORES_MAX, auto_nsplit, tile_nsplit
    for T in (64, 72, 100, 127, 128, 144, 170):
        for keys in (4096, 8192, 43680):
            split, need = auto_nsplit(T, keys, HD)
            if T * keys * 32 <= SCORES_MAX:
                assert split == 512 // T >= 3 and need == T * keys * 32
            else:
                assert (split, need) == (tile_nsplit(T, keys), 0)
    for keys in (2064, 4096):
        assert auto_nsplit(128, keys, HD)[1] > 0
        for T in (1, 8, 40, 63, 171, 176, 184, 256, 512, 1024, 2048):
            assert auto_nsplit(T, keys, HD) == (tile_nsplit(T, keys), 0), (T, keys)
    for T in (128, 144, 160, 176, 184, 191, 192):
        for keys in (16, 1024, 2032, 2048):
            assert auto_nsplit(T, keys, HD) == (1, 0), (T, keys)


def test_grouped_rule():
    """The grouped form from its number of (token, KV head)s and of tokens per table row on, never past its scratch."""
    from bitexact.vllm_plugin.tri_exact_attn import rows_scratch
    for HD, tokens in ((64, 192), (128, 144)):
        for HKV in (1, 8):
            t = tokens * 8 // HKV
            assert rows_scratch(t, HKV, 4, HD, 8, 512) > 0 and rows_scratch(t - 1, HKV, 4, HD, 8, 512) == 0
        assert rows_scratch(8 * 40, 8, 4, HD, 40, 512) > 0 and rows_scratch(8 * 40 - 1, 8, 4, HD, 40, 512) == 0
        assert rows_scratch(4096, 8, 4, HD, 64, 16384) == 0
        assert rows_scratch(4096, 8, 4, HD, 8, 43700) == rows_scratch(4096, 8, 5, HD, 8, 512) == 0
    assert rows_scratch(4096, 8, 4, 96, 8, 512) == 0
