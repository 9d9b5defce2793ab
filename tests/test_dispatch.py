"""Which form the attention entry points choose by size (no GPU call is made)."""

import ctypes

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


def test_int8_tile_plan():
    """The int8 product's plan names the kernel that is launched and asks for that kernel's workspace: the pipelined
    tiles (6) on both sides of their number of tiles at short, middle and long K, each with its waves; else the tile
    kernel (3), which splits K."""
    from bitexact import _hip
    L = _hip.lib()
    out = (ctypes.c_int32 * 6)()

    def plan(M, N, K, nl):
        assert L.bx_int8_gemm_plan(M, N, K, nl, out) == 0
        ws = L.bx_int8_gemm_workspace(M, N, K, max(nl, 1))
        assert (ws > 0) == (out[2] > 1)
        return tuple(out[:4])
    bn, bm = {0: 256, 1: 256, 2: 128, 3: 128}, {0: 128, 1: 128, 2: 128, 3: 64}
    for nl in (0, 1, 2, 3):
        for K, line in ((64, 8), (2048, 8), (2112, 24), (4096, 24)):
            M, N = 4 * bm[nl], line // 4 * bn[nl]          # four row tiles
            assert plan(M, N, K, nl) == (6, 4, 1, line), (nl, K)
            kernel, tile, split, blocks = plan(M, N - bn[nl], K, nl)
            assert kernel == 3 and tile != 4 and blocks > 0, (nl, K)
            assert plan(M, N, K + 16, nl)[0] == 3
    for K in (4160, 8192):                                 # by the tile kernel's 64 x 128 tiles
        assert plan(512, 2048, K, 2)[0] == 6 and plan(448, 2048, K, 2)[0] == 3 and plan(400, 2048, K, 2)[0] == 3
        assert plan(384, 2048, K, 3)[0] == 6 and plan(320, 2048, K, 3)[0] == 3
    # one limb where the tile kernel runs unsplit
    for K, M in ((64, 1024), (2048, 1024), (2112, 1280), (4096, 1280), (8192, 1280)):
        assert plan(M, 2048, K, 1)[:3] == (6, 4, 1) and plan(M - 128, 2048, K, 1)[::2] == (3, 1), K
        assert plan(1792, 2047, K, 0)[:3] == (6, 4, 1) and plan(1664, 2047, K, 1)[::2] == (3, 1), K
    assert plan(256, 2048, 8192, 1)[0] == 3                # a split, past K = 4096
    assert plan(2048, 16384, 2048, 1) == (6, 4, 1, 16 * 64)
    assert plan(2048, 16384, 2048, 2) == plan(2048, 16384, 2048, 3) == (6, 8, 1, 16 * 64)
    assert plan(1024, 4096, 4096, 2) == (6, 4, 1, 8 * 32) and plan(1500, 4096, 4096, 2) == (6, 8, 1, 12 * 16)
    assert plan(704, 16384, 2048, 3) == (6, 4, 1, 11 * 128) and plan(705, 16384, 2048, 3) == (6, 8, 1, 6 * 64)
    assert plan(2048, 1 << 20, 2048, 1)[0] == 3            # weights past the 32-bit offsets
