"""HIP attention-side kernels against the CPU oracle, bit for bit: paged exact attention (reference
tests/test_vllm_exact_attn.py: head_dim 64 / 128, three magnitudes, five (R, M, P) cases, four splits),
the paged KV store, the fused prefill attention (exact/model.py's bmm -> softmax -> bmm), and the limb bmm
(reference tests/test_gpu_kernels.py:9-19)."""

import numpy as np
import pytest
import torch

from oracle import bxref as R

pytestmark = pytest.mark.gpu


def _lut(dev):
    return torch.from_numpy(R.exp2_table()).to(dev)


def test_kv_store_matches_oracle(dev):
    from bitexact.vllm_plugin.tri_paged import store, to_limbs
    g = torch.Generator().manual_seed(0)
    c = torch.randint(-R.LIM3, R.LIM3 + 1, (5, 3, 16, 2 * 64), generator=g).to(torch.int32)
    assert np.array_equal(to_limbs(c.to(dev)).cpu().numpy(), R.to_limbs(c.numpy()))
    # store with skipped slots and int64 input
    cache = torch.zeros(4, 2, 16, 8 * 64, dtype=torch.int8, device=dev)
    k = torch.randint(-R.LIM3, R.LIM3 + 1, (6, 2, 64), generator=g)
    v = torch.randint(-R.LIM3, R.LIM3 + 1, (6, 2, 64), generator=g)
    slot = torch.tensor([0, 17, -1, 33, 63, 5])
    store(cache, slot.to(dev), k.to(dev), v.to(dev))
    ref = np.zeros((4, 2, 16, 8 * 64), np.int8)
    kv = np.concatenate([k.numpy(), v.numpy()], -1)
    lim = R.to_limbs(kv[:, :, None, :].transpose(0, 1, 2, 3).reshape(6, 2, 1, 128))
    for n, s in enumerate(slot.tolist()):
        if s >= 0:
            ref[s // 16, :, s % 16] = lim[n, :, 0]
    assert np.array_equal(cache.cpu().numpy(), ref)


@pytest.mark.parametrize("HD", [64, 128])
def test_exact_paged_attention(dev, HD):
    from bitexact.vllm_plugin import tri_exact_attn, tri_paged
    g = torch.Generator().manual_seed(HD)
    lut = _lut(dev)
    nb, bs, HKV = 96, 16, 8
    l2e = R.L2E28_HD[HD]
    for lim in (R.LIM3, 1 << 13, 1 << 10):
        c = torch.randint(-lim, lim + 1, (nb, HKV, bs, 2 * HD), generator=g).to(torch.int32)
        cl = tri_paged.to_limbs(c.to(dev))
        for Rr, M, P in [(3, 4, 600), (5, 4, 3000), (6, 1, 900), (2, 3, 50), (7, 4, 5)]:
            bt = torch.randint(1, nb, (Rr, 200), generator=g).to(torch.int32)
            qpos = torch.randint(0, P, (Rr, M), generator=g)
            q = torch.randint(-(1 << 22), (1 << 22) + 1, (Rr, HKV, M, HD), generator=g).to(torch.int32)
            sh = torch.randint(-40, -10, (Rr, HKV, M), generator=g)
            rmap = torch.arange(Rr)
            ref_num, ref_den = R.paged_attend(q.numpy(), sh.numpy(), qpos.numpy(), c.numpy(), bt.numpy(),
                                              rmap.numpy(), R.exp2_table(), l2e)
            for ns in (None, 1, 5, 64):
                num, den = tri_exact_attn.attend(q.to(dev), sh.to(dev), qpos.to(dev), cl, bt.to(dev), rmap.to(dev),
                                                 lut, l2e, nsplit=ns)
                assert np.array_equal(num.cpu().numpy(), ref_num), (Rr, M, ns, lim)
                assert np.array_equal(den.cpu().numpy(), ref_den), (Rr, M, ns, lim)


def test_paged_attention_rmap_and_empty_rows(dev):
    """Rows mapped to shared block-table rows, a query with no visible key (qpos -1), repeated calls
    (the split workspace is restored after each call)."""
    from bitexact.vllm_plugin import tri_exact_attn, tri_paged
    g = torch.Generator().manual_seed(7)
    HD, nb, bs, HKV = 64, 20, 16, 2
    c = torch.randint(-R.LIM3, R.LIM3 + 1, (nb, HKV, bs, 2 * HD), generator=g).to(torch.int32)
    cl = tri_paged.to_limbs(c.to(dev))
    bt = torch.randint(0, nb, (2, 8), generator=g).to(torch.int32)
    rmap = torch.tensor([1, 0, 1])
    qpos = torch.tensor([[100, -1, 3, 127], [5, 6, 7, 8], [0, 0, 0, 0]])
    q = torch.randint(-(1 << 22), (1 << 22) + 1, (3, HKV, 4, HD), generator=g).to(torch.int32)
    sh = torch.randint(-40, -10, (3, HKV, 4), generator=g)
    ref = R.paged_attend(q.numpy(), sh.numpy(), qpos.numpy(), c.numpy(), bt.numpy(), rmap.numpy(), R.exp2_table(),
                         R.L2E28)
    for ns in (3, 3, 1, 8):
        num, den = tri_exact_attn.attend(q.to(dev), sh.to(dev), qpos.to(dev), cl, bt.to(dev), rmap.to(dev), _lut(dev),
                                         R.L2E28, nsplit=ns)
        assert np.array_equal(num.cpu().numpy(), ref[0]) and np.array_equal(den.cpu().numpy(), ref[1]), ns


@pytest.mark.parametrize("HD,bs,nblk,M", [(64, 16, 128, 4), (128, 4, 300, 3), (64, 1, 700, 1), (128, 16, 9, 2)])
def test_paged_attention_one_block_per_tile(dev, HD, bs, nblk, M):
    """The unsplit launch for rows of at most 2048 keys (block-table row copied to LDS, scores kept in LDS, K and V
    streamed once through a register ring): cache blocks of 16, 4 and 1 keys, the full 2048-key reach, queries
    past nvalid, a query with no visible key; against the oracle."""
    from bitexact.vllm_plugin import tri_exact_attn, tri_paged
    g = torch.Generator().manual_seed(HD + bs + nblk)
    HKV, Rr = 2, 3
    nb = Rr * nblk + 1
    c = torch.randint(-R.LIM3, R.LIM3 + 1, (nb, HKV, bs, 2 * HD), generator=g).to(torch.int32)
    cl = tri_paged.to_limbs(c.to(dev))
    bt = (1 + torch.randperm(Rr * nblk, generator=g)).to(torch.int32).reshape(Rr, nblk)
    S = nblk * bs
    qpos = torch.randint(0, S, (Rr, M), generator=g)
    qpos[0, 0] = S - 1
    if M > 1:
        qpos[1, 1] = -1
    q = torch.randint(-(1 << 22), (1 << 22) + 1, (Rr, HKV, M, HD), generator=g).to(torch.int32)
    sh = torch.randint(-40, -10, (Rr, HKV, M), generator=g)
    rmap = torch.tensor([2, 0, 1])
    l2e = R.L2E28_HD[HD]
    ref = R.paged_attend(q.numpy(), sh.numpy(), qpos.numpy(), c.numpy(), bt.numpy(), rmap.numpy(), R.exp2_table(),
                         l2e)
    num, den = tri_exact_attn.attend(q.to(dev), sh.to(dev), qpos.to(dev), cl, bt.to(dev), rmap.to(dev), _lut(dev),
                                     l2e, nsplit=1)
    assert np.array_equal(num.cpu().numpy(), ref[0]) and np.array_equal(den.cpu().numpy(), ref[1])


@pytest.mark.parametrize("ticks,ns", [(None, 8), ("0", 8), (None, 4), ("0", 4)])
def test_paged_attention_split_exchange(dev, monkeypatch, ticks, ns):
    """Config 4's decode shape (4 rows x 8 KV heads, 2048 keys, group 4) over 8 or 4 key splits in one launch, where the
    splits of a tile exchange their maxima through the workspace: equal to the unsplit launch and to the oracle on
    a sample of tiles, three calls in a row. ticks "0": no wait for the other splits, each block computes the
    maxima it has not seen from the keys (the path a block takes when its partners are not resident)."""
    from bitexact.vllm_plugin import tri_exact_attn, tri_paged
    if ticks is not None:
        monkeypatch.setenv("BX_ATTN_EXCH_TICKS", ticks)
    g = torch.Generator().manual_seed(11)
    B, HKV, M, HD, S, bs = 4, 8, 4, 64, 2048, 16
    nblk = S // bs
    c = torch.randint(-R.LIM3, R.LIM3 + 1, (B * nblk, HKV, bs, 2 * HD), generator=g).to(torch.int32)
    cl = tri_paged.to_limbs(c.to(dev))
    bt = torch.randperm(B * nblk, generator=g).to(torch.int32).reshape(B, nblk)
    qpos = torch.tensor([[S - 1] * M, [S - 1, 1000, 5, 0], [1500] * M, [2047, 2046, 64, 63]])
    q = torch.randint(-(1 << 22), (1 << 22) + 1, (B, HKV, M, HD), generator=g).to(torch.int32)
    sh = torch.randint(-40, -25, (B, HKV, M), generator=g)
    args = (q.to(dev), sh.to(dev), qpos.to(dev), cl, bt.to(dev), torch.arange(B).to(dev), _lut(dev), R.L2E28)
    assert tri_exact_attn.default_nsplit(B, HKV, nblk, bs) == 8
    n1, d1 = tri_exact_attn.attend(*args, nsplit=1)
    for _ in range(3):
        n8, d8 = tri_exact_attn.attend(*args, nsplit=ns)
        assert torch.equal(n8, n1) and torch.equal(d8, d1)
    rows = [0, 1]
    ref_num, ref_den = R.paged_attend(q[rows].numpy(), sh[rows].numpy(), qpos[rows].numpy(), c.numpy(),
                                      bt[rows].numpy(), np.arange(2), R.exp2_table(), R.L2E28)
    assert np.array_equal(n8[:2].cpu().numpy(), ref_num) and np.array_equal(d8[:2].cpu().numpy(), ref_den)


@pytest.mark.parametrize("HD", [64, 128])
@pytest.mark.parametrize("planes,shr", [(True, (-40, -10)), (False, (-40, -10)), (True, (-9, 7))])
def test_prefill_attention(dev, HD, planes, shr):
    """Both prefill forms (limb planes streamed into LDS; register-staged) against the oracle's unfused
    bmm -> softmax -> bmm, on a strided cache view with two sequence offsets. Query exponents from -9 up give
    negative score shifts for some rows (the limb-plane kernel's general weight path)."""
    from bitexact.exact.attention import prefill
    g = torch.Generator().manual_seed(3 + HD)
    B, HKV, grp, T, L = 2, 2, 4, 70, 96
    Z = B * HKV
    qg = torch.randint(-(1 << 22), (1 << 22) + 1, (Z, grp * T, HD), generator=g).to(torch.int32)
    shg = torch.randint(shr[0], shr[1], (Z, grp * T, 1), generator=g)
    cache_k = torch.randint(-R.LIM3, R.LIM3 + 1, (B, HKV, L, HD), generator=g).to(torch.int32)
    cache_v = torch.randint(-R.LIM3, R.LIM3 + 1, (B, HKV, L, HD), generator=g).to(torch.int32)
    pos = torch.arange(T)[None].expand(B, T) + torch.tensor([[0], [20]])           # two sequences, offsets
    S = int(pos.max()) + 1
    qpos = pos[:, None, None, :].expand(B, HKV, grp, T).reshape(Z, grp * T, 1)
    Kc = cache_k[:, :, :S].reshape(Z, S, HD)
    Vc = cache_v[:, :, :S].reshape(Z, S, HD)
    ref_num, ref_den = R.attention_prefill(qg.numpy(), shg.numpy(), Kc.numpy(), Vc.numpy(), qpos.numpy(),
                                           R.exp2_table(), R.L2E28_HD[HD])
    kd = cache_k.to(dev)[:, :, :S].reshape(Z, S, HD)      # strided view of the cache (row stride L * HD)
    vd = cache_v.to(dev)[:, :, :S].reshape(Z, S, HD)
    num, den = prefill(qg.to(dev), shg.to(dev), kd, vd, qpos.to(dev), _lut(dev), R.L2E28_HD[HD], planes=planes)
    assert np.array_equal(num.cpu().numpy(), ref_num) and np.array_equal(den.cpu().numpy(), ref_den)


@pytest.mark.parametrize("HD,T,Z", [(64, 2048, 4), (128, 640, 2)])
def test_prefill_attention_full_size(dev, HD, T, Z):
    """Config 4's prefill shape (group 4, causal T = 2048) and a head_dim-128 case: the limb-plane form equals the
    register-staged form on every row (two kernels with different tilings and operand orders), every row that
    sees a key has den >= 2^22 (its own maximum's weight is 2^FP), and a sample of rows (first and last of each
    head's block, the partial last tile) equals the oracle."""
    from bitexact.exact.attention import prefill
    g = torch.Generator().manual_seed(HD + T)
    grp = 4
    qg = torch.randint(-(1 << 22), (1 << 22) + 1, (Z, grp * T, HD), generator=g).to(torch.int32)
    shg = torch.randint(-40, -25, (Z, grp * T, 1), generator=g)
    K = torch.randint(-R.LIM3, R.LIM3 + 1, (Z, T, HD), generator=g).to(torch.int32)
    V = torch.randint(-R.LIM3, R.LIM3 + 1, (Z, T, HD), generator=g).to(torch.int32)
    qpos = torch.arange(T).repeat(grp).reshape(1, grp * T, 1).expand(Z, grp * T, 1).contiguous()
    args = (qg.to(dev), shg.to(dev), K.to(dev), V.to(dev), qpos.to(dev), _lut(dev), R.L2E28_HD[HD])
    n1, d1 = prefill(*args, planes=True)
    n2, d2 = prefill(*args, planes=False)
    assert torch.equal(n1, n2) and torch.equal(d1, d2)
    assert bool((d1 >= 1 << 22).all())
    rows = np.unique(np.concatenate([np.arange(0, 40), np.arange(T - 40, T + 40), np.arange(grp * T - 70, grp * T)]))
    z = Z - 1
    ref_num, ref_den = R.attention_prefill(qg[z:z + 1, rows].numpy(), shg[z:z + 1, rows].numpy(), K[z:z + 1].numpy(),
                                           V[z:z + 1].numpy(), qpos[z:z + 1, rows].numpy(), R.exp2_table(),
                                           R.L2E28_HD[HD])
    assert np.array_equal(n1[z, rows].cpu().numpy(), ref_num[0]) and np.array_equal(d1[z, rows].cpu().numpy(),
                                                                                     ref_den[0])


@pytest.mark.parametrize("mode", ["exact", "int8"])
@pytest.mark.parametrize("HD,Rr,M,keys", [(64, 16, 4, 2064), (64, 8, 3, 4096), (128, 16, 1, 2064), (128, 9, 4, 4112),
                                            (64, 21, 2, 3072)])
def test_paged_kept_scores(dev, mode, HD, Rr, M, keys):
    """Long contexts keep the scores between their two launches (attend chooses that by size): equal to the one-launch
    or K-twice forms on every row, with contexts that end anywhere in the table (one key, a split's first and last
    key, none, the longest that one block takes alone and one more), and repeated (the workspace is left zero)."""
    from bitexact.int8.consts import exp_table
    from bitexact.vllm_plugin import tri_exact_attn, tri_paged
    g = torch.Generator().manual_seed(keys)
    HKV, bs = 8, 16
    nblk = keys // bs
    tiles = Rr * HKV
    split, need = tri_exact_attn.auto_nsplit(tiles, keys, HD)
    assert need > 0 and split > 1
    lim = R.LIM3 if mode == "exact" else 1 << 14
    cl = tri_paged.to_limbs(torch.randint(-lim, lim + 1, (Rr * nblk, HKV, bs, 2 * HD), generator=g).to(torch.int32).to(dev))
    bt = torch.randperm(Rr * nblk, generator=g).to(torch.int32).view(Rr, nblk).to(dev)
    qpos = torch.full((Rr, M), keys - 1)
    one = 256 * 64 // HD
    ends = [0, 1, 63, 64, keys // split - 1, keys // split, keys - 2, -1, one - 1, one, one - 17]
    for i, e in enumerate(ends[:Rr]):
        qpos[i] = e
    qpos[3, 0] = 700
    qpos = qpos.to(dev)
    if mode == "exact":
        q = torch.randint(-(1 << 22), (1 << 22) + 1, (Rr, HKV, M, HD), generator=g).to(torch.int32).to(dev)
        sh = torch.randint(-44, -36, (Rr, HKV, M), generator=g).to(dev)
        run = lambda **k: tri_exact_attn.attend(q, sh, qpos, cl, bt, torch.arange(Rr, device=dev), _lut(dev),
                                                R.L2E28_HD[HD], **k)
    else:
        q = torch.randint(-(1 << 15), (1 << 15) + 1, (Rr, HKV, M, HD), generator=g).to(dev)
        ptab = tri_paged.weight_table(exp_table(dev))
        run = lambda **k: tri_paged.attend(q, qpos, cl, bt, ptab, **k)
    n1, d1 = run(nsplit=1)
    for _ in range(3):
        n2, d2 = run()
        assert torch.equal(n1, n2) and torch.equal(d1, d2)


@pytest.mark.parametrize("HD,M,bs", [(64, 4, 16), (64, 3, 16), (64, 1, 32), (128, 4, 16), (128, 2, 16)])
@pytest.mark.parametrize("order", ["runs", "mixed"])
def test_paged_rows_equal_decode_form(dev, HD, M, bs, order):
    """attend's grouped form (prefill steps) against the per-token form, bit for bit: sequences whose token counts are
    at a tile's edges (0, 1, one short of a tile, a tile, one over, several), chunks that start past other keys,
    padding tokens (position -1), the tokens of a sequence in a row or all mixed, strided cache heads."""
    from bitexact.vllm_plugin import tri_exact_attn, tri_paged
    g = torch.Generator().manual_seed(HD + M)
    HKV, TT = 2, (128 if HD == 64 else 64) // M
    counts, start = [0, 1, TT - 1, TT, TT + 1, 1200, 70], [0, 300, 5, 64, 63, 0, 129]
    nrow, nblk = len(counts), -(-(max(s + n for s, n in zip(start, counts))) // bs)
    c = torch.randint(-R.LIM3, R.LIM3 + 1, (nrow * nblk, HKV, bs, 2 * HD), generator=g).to(torch.int32)
    cl = tri_paged.to_limbs(c.to(dev))
    bt = torch.randperm(nrow * nblk, generator=g).to(torch.int32).view(nrow, nblk).to(dev)
    rmap = torch.cat([torch.full((n,), i) for i, n in enumerate(counts)])
    pos = torch.cat([torch.arange(n) + s for s, n in zip(start, counts)])
    if order == "mixed":
        p = torch.randperm(len(pos), generator=g)
        rmap, pos = rmap[p], pos[p]
    pos[::17] = -1
    Rr = len(pos)
    qpos = pos[:, None].expand(Rr, M).contiguous()
    q = torch.randint(-(1 << 22), (1 << 22) + 1, (Rr, HKV, M, HD), generator=g).to(torch.int32)
    sh = torch.randint(-46, -36, (Rr, HKV, M), generator=g)
    args = (q.to(dev), sh.to(dev), qpos.to(dev), cl, bt, rmap.to(dev), _lut(dev), R.L2E28_HD[HD])
    assert tri_exact_attn.rows_scratch(Rr, HKV, M, HD, nrow, nblk * bs) > 0
    n1, d1 = tri_exact_attn.attend(*args, nsplit=1)
    for _ in range(2):
        n2, d2 = tri_exact_attn.attend(*args)
        assert torch.equal(n1, n2) and torch.equal(d1, d2)


@pytest.mark.parametrize("HD,HKV,M,keys,few,chunks", [
    (64, 4, 4, 2048, [7, 8, 9, 1, 0, 6], [300, 130]),          # the line; few rows: many splits
    (128, 4, 3, 4096, [1] * 20 + [7], [400]),
    (64, 4, 4, 640, [7] * 40 + [3] * 20, [260, 1]),            # more tiles than blocks: one split
    (128, 4, 2, 1024, [5] * 11 + [8], [250]),                  # 220 tiles: two splits
    (64, 8, 4, 16384, [1] * 15, [200]),                        # scores past their limit: K read twice
    (128, 8, 1, 16384, [7] * 3 + [1] * 6, [150])])
def test_paged_rows_mixed_steps(dev, HD, HKV, M, keys, few, chunks):
    """Steps of prefill chunks and sequences with few tokens (decoding ones) in the grouped form against the per-token
    form, bit for bit: counts at the line between the two, contexts of any length (none, one key, the last), tokens of a
    sequence in any order, padding rows outside the table, repeated on the same scratch."""
    from bitexact.vllm_plugin import tri_exact_attn, tri_paged
    g = torch.Generator().manual_seed(HD + keys + len(few))
    bs, nphys = 16, 96
    nblk, counts = keys // bs, few + chunks
    nrow = len(counts)
    c = torch.randint(-R.LIM3, R.LIM3 + 1, (nphys, HKV, bs, 2 * HD), generator=g).to(torch.int32)
    cl = tri_paged.to_limbs(c.to(dev))
    bt = torch.randint(0, nphys, (nrow, nblk), generator=g).to(torch.int32).to(dev)
    rmap = torch.cat([torch.full((n,), i) for i, n in enumerate(counts)])
    rmap = rmap[torch.randperm(len(rmap), generator=g)]
    Rr = len(rmap)
    qpos = torch.randint(-1, keys, (Rr, M), generator=g)
    qpos[::5] = torch.randint(-1, 300, (len(qpos[::5]), 1), generator=g)
    qpos[1], qpos[2], qpos[3] = keys - 1, 0, -1
    inside = torch.ones(Rr, dtype=torch.bool)
    inside[7::31] = False
    q = torch.randint(-(1 << 22), (1 << 22) + 1, (Rr, HKV, M, HD), generator=g).to(torch.int32).to(dev)
    sh = torch.randint(-46, -36, (Rr, HKV, M), generator=g).to(dev)
    args = lambda r, p: (q, sh, p.to(dev), cl, bt, r.to(dev), _lut(dev), R.L2E28_HD[HD])
    assert tri_exact_attn.rows_scratch(Rr, HKV, M, HD, nrow, keys) > 0
    n1, d1 = tri_exact_attn.attend(*args(rmap, torch.where(inside[:, None], qpos, -1)), nsplit=1)
    for _ in range(3):
        n2, d2 = tri_exact_attn.attend(*args(torch.where(inside, rmap, nrow), qpos))
        assert torch.equal(n1, n2) and torch.equal(d1, d2)


@pytest.mark.parametrize("HD", [64, 128])
def test_positions_below_int32_see_no_key(dev, HD):
    """Rows masked by a position of any negative value (the type's lowest, low words that read as a position) see no
    key, as with -1: the grouped paged form against the per-token one, and the limb-plane prefill."""
    from bitexact.exact.attention import prefill
    from bitexact.vllm_plugin import tri_exact_attn, tri_paged
    g = torch.Generator().manual_seed(HD)
    HKV, M, bs, nrow, nblk, Rr = 4, 4, 16, 3, 12, 400
    S = nblk * bs
    c = torch.randint(-R.LIM3, R.LIM3 + 1, (nrow * nblk, HKV, bs, 2 * HD), generator=g).to(torch.int32)
    cl = tri_paged.to_limbs(c.to(dev))
    bt = torch.randperm(nrow * nblk, generator=g).to(torch.int32).view(nrow, nblk).to(dev)
    rmap = torch.randint(0, nrow, (Rr,), generator=g).to(dev)
    low = torch.tensor([-(1 << 63), -(1 << 32), 100 - (1 << 40), -(1 << 31) - 1, -1])
    masked = torch.rand(Rr, M, generator=g) < 0.5
    masked[rmap.cpu() == 0] = True                         # a sequence without any visible key
    qpos = torch.randint(0, S, (Rr, M), generator=g)
    lowest = low[torch.randint(0, len(low), (Rr, M), generator=g)]
    q = torch.randint(-(1 << 22), (1 << 22) + 1, (Rr, HKV, M, HD), generator=g).to(torch.int32).to(dev)
    sh = torch.randint(-46, -36, (Rr, HKV, M), generator=g).to(dev)
    assert tri_exact_attn.rows_scratch(Rr, HKV, M, HD, nrow, S) > 0
    run = lambda p, ns: tri_exact_attn.attend(q, sh, p.to(dev), cl, bt, rmap, _lut(dev), R.L2E28_HD[HD], nsplit=ns)
    (n1, d1), (n2, d2) = run(torch.where(masked, -1, qpos), 1), run(torch.where(masked, lowest, qpos), None)
    assert torch.equal(n1, n2) and torch.equal(d1, d2)
    Z, gT = 2, M * 100
    K, V = (torch.randint(-R.LIM3, R.LIM3 + 1, (Z, S, HD), generator=g).to(torch.int32).to(dev) for _ in range(2))
    qz, shz = q.view(-1, HD)[:Z * gT].view(Z, gT, HD), sh.view(-1)[:Z * gT].view(Z, gT, 1)
    pz = lambda p: p.view(-1)[:Z * gT].view(Z, gT, 1).to(dev)
    (n1, d1), (n2, d2) = (prefill(qz, shz, K, V, pz(torch.where(masked, m, qpos)), _lut(dev), R.L2E28_HD[HD])
                          for m in (torch.tensor(-1), lowest))
    assert torch.equal(n1, n2) and torch.equal(d1, d2)


@pytest.mark.parametrize("HD,npad,pad", [(64, 1, -1), (64, 33, -1), (64, 300, -(1 << 40)), (128, 40, 3), (128, 200, 1 << 40),
                                         (64, 513, None)])
def test_paged_rows_outside_the_table(dev, HD, npad, pad):
    """Tokens whose rmap names no table row (negative, nrow, beyond; None: all of them mixed) in a step that takes the
    grouped form: their num and den are 0 and the other tokens' are the per-token form's. The counts cover a tile's
    edges (32 tokens of 4 queries at heads of 64, 16 at 128), and scratch holds another step's slots before the call."""
    from bitexact import _hip
    from bitexact.vllm_plugin import tri_exact_attn, tri_paged
    g = torch.Generator().manual_seed(HD + npad)
    HKV, M, bs, nrow, nblk = 4, 4, 16, 3, 12
    c = torch.randint(-R.LIM3, R.LIM3 + 1, (nrow * nblk, HKV, bs, 2 * HD), generator=g).to(torch.int32)
    cl = tri_paged.to_limbs(c.to(dev))
    bt = torch.randperm(nrow * nblk, generator=g).to(torch.int32).view(nrow, nblk).to(dev)
    Rr = 400 + npad
    live = torch.ones(Rr, dtype=torch.bool)
    live[torch.randperm(Rr, generator=g)[:npad]] = False
    rmap = torch.randint(0, nrow, (Rr,), generator=g)
    qpos = torch.randint(-1, nblk * bs, (Rr, M), generator=g)
    q = torch.randint(-(1 << 22), (1 << 22) + 1, (Rr, HKV, M, HD), generator=g).to(torch.int32).to(dev)
    sh = torch.randint(-46, -36, (Rr, HKV, M), generator=g).to(dev)
    args = lambda r, p: (q, sh, p.to(dev), cl, bt, r.to(dev), _lut(dev), R.L2E28_HD[HD])
    n1, d1 = tri_exact_attn.attend(*args(rmap, torch.where(live[:, None], qpos, -1)), nsplit=1)
    outside = torch.tensor([-1, nrow, 1 << 40, -(1 << 40), (1 << 32) + 1])
    fill = torch.full((Rr,), pad) if pad is not None else outside[torch.randint(0, len(outside), (Rr,), generator=g)]
    need = tri_exact_attn.rows_scratch(Rr, HKV, M, HD, nrow, nblk * bs)
    assert need > 0
    _hip.scratch(dev, need)[0].fill_(1)
    n2, d2 = tri_exact_attn.attend(*args(torch.where(live, rmap, fill), qpos))
    assert torch.equal(n1, n2) and torch.equal(d1, d2)


@pytest.mark.parametrize("HD", [64, 128])
@pytest.mark.parametrize("table", ["exp2", "noisy", "steps"])
def test_prefill_weight_positions(dev, HD, table):
    """The limb-plane form's short weight rule at the table positions where it can go wrong, against the oracle:
    scores placed one by one (z = max - raw exactly, shift 0) on both sides of every integer n (the weight's binade
    changes, n = 22 / 23 where it becomes 1 and 0), at table entries, and 1400 positions in the first three binades
    (a few of them within the 32-bit table's uncertainty of a rounding boundary). "noisy": a table whose entries are
    off by more than its float64 factors allow; "steps": one outside [2^59, 2^60]; both take the general rule."""
    from bitexact.exact.attention import prefill
    l2e = R.L2E28_HD[HD]
    rng = np.random.default_rng(HD)
    lut = R.exp2_table().copy()
    if table == "noisy":
        lut[1:-1] += rng.integers(-(1 << 20), 1 << 20, len(lut) - 2)
    elif table == "steps":
        lut = (lut >> 3) << 2
    zf = [0]
    for n in range(27):
        for f in (0, 1, 4095, 4096, 1 << 25):
            z0 = (((n << 26) + f) << 28) // l2e
            zf += [z0 - 1, z0, z0 + 1, z0 + 2]
    zf = np.concatenate([np.clip(np.array(zf, dtype=np.int64), 0, None), rng.integers(0, 3 << 26, 1400)])
    rng.shuffle(zf)
    S, T, Z = len(zf), 70, 1
    K = np.zeros((Z, S, HD), np.int64)
    K[0, :, 0], K[0, :, 1] = (-zf) >> 20, (-zf) & ((1 << 20) - 1)     # raw = 2^20 K0 + K1 = -zf
    V = rng.integers(-R.LIM3, R.LIM3 + 1, (Z, S, HD))
    q = np.zeros((Z, T, HD), np.int64)
    q[0, :, 0], q[0, :, 1] = 1 << 20, 1
    sh = np.full((Z, T, 1), -6)                                        # shift FK + 3 - FZ - sh = 0
    qpos = np.sort(rng.integers(0, S, (Z, T, 1)), axis=1)
    ref_num, ref_den = R.attention_prefill(q, sh, K, V, qpos, lut, l2e)
    t32 = lambda x: torch.from_numpy(x).to(torch.int32).to(dev)
    num, den = prefill(t32(q), torch.from_numpy(sh).to(dev), t32(K), t32(V), torch.from_numpy(qpos).to(dev),
                       torch.from_numpy(lut).to(dev), l2e)
    assert np.array_equal(den.cpu().numpy(), ref_den) and np.array_equal(num.cpu().numpy(), ref_num)


@pytest.mark.parametrize("HD,T", [(64, 1), (64, 31), (64, 33), (128, 15), (128, 17), (64, 65)])
def test_prefill_row_tiles(dev, HD, T):
    """Row tiles at their edges (128 rows at head_dim 64, 64 at 128; 4 T rows) with key tiles whole, one short and
    one over, rows that see no key (position -1) among them, against the register-staged form."""
    from bitexact.exact.attention import prefill
    g = torch.Generator().manual_seed(T)
    Z, S = 3, T + 63
    qg = torch.randint(-(1 << 22), (1 << 22) + 1, (Z, 4 * T, HD), generator=g).to(torch.int32).to(dev)
    shg = torch.randint(-24, -18, (Z, 4 * T, 1), generator=g).to(dev)
    K = (torch.randn(Z, S, HD, generator=g) * 2 ** 17).to(torch.int32).to(dev)
    V = torch.randint(-R.LIM3, R.LIM3 + 1, (Z, S, HD), generator=g).to(torch.int32).to(dev)
    qpos = torch.randint(-1, S, (Z, 4 * T, 1), generator=g).to(dev)
    args = (qg, shg, K, V, qpos, _lut(dev), R.L2E28_HD[HD])
    n1, d1 = prefill(*args, planes=True)
    n2, d2 = prefill(*args, planes=False)
    assert torch.equal(n1, n2) and torch.equal(d1, d2)


def test_bmm_exact(dev):
    from bitexact.bmm import bmm
    g = torch.Generator().manual_seed(0)
    # (two 64-row tiles per block from M = 128; one k step when K <= 64)
    for Z, M, K, N in [(3, 5, 64, 70), (16, 4, 700, 64), (2, 130, 64, 129), (2, 70, 33, 600), (2, 200, 33, 300),
                       (2, 256, 700, 64)]:
        a = torch.randint(-R.LIM3, R.LIM3 + 1, (Z, M, K), generator=g)
        b = torch.randint(-R.LIM3, R.LIM3 + 1, (Z, K, N), generator=g).to(torch.int32)
        ref = R.bmm(a.numpy(), b.numpy())
        assert np.array_equal(bmm(a.to(dev), b.to(dev)).cpu().numpy(), ref)
        bt = b.to(dev).transpose(1, 2).contiguous().transpose(1, 2)
        assert np.array_equal(bmm(a.to(dev), bt).cpu().numpy(), ref)
    # fewer limbs: values within 1 limb times 3-limb values
    a = torch.randint(-128, 128, (2, 9, 33), generator=g)
    b = torch.randint(-R.LIM3, R.LIM3 + 1, (2, 33, 11), generator=g)
    assert np.array_equal(bmm(a.to(dev), b.to(dev), na=1).cpu().numpy(), R.bmm(a.numpy(), b.numpy()))
    for na, nb in ((1, 2), (2, 3), (3, 1), (2, 2)):
        la, lb = (-128, 127) if na == 1 else (-R.LIM[na], R.LIM[na]), (-128, 127) if nb == 1 else (-R.LIM[nb], R.LIM[nb])
        a = torch.randint(la[0], la[1] + 1, (3, 70 if na != 2 else 150, 150), generator=g)
        b = torch.randint(lb[0], lb[1] + 1, (3, 150, 66), generator=g)
        assert np.array_equal(bmm(a.to(dev), b.to(dev), na=na, nb=nb).cpu().numpy(), R.bmm(a.numpy(), b.numpy()))
    # A transposed in memory (m contiguous), both int32
    a = torch.randint(-R.LIM3, R.LIM3 + 1, (2, 67, 100), generator=g).to(torch.int32)
    b = torch.randint(-R.LIM3, R.LIM3 + 1, (2, 100, 65), generator=g).to(torch.int32)
    at = a.to(dev).transpose(1, 2).contiguous().transpose(1, 2)
    assert np.array_equal(bmm(at, b.to(dev)).cpu().numpy(), R.bmm(a.numpy(), b.numpy()))
    for M, K in ((190, 100), (129, 40)):   # the same over two row tiles per block
        a = torch.randint(-R.LIM3, R.LIM3 + 1, (2, M, K), generator=g).to(torch.int32)
        b = torch.randint(-R.LIM3, R.LIM3 + 1, (2, K, 65), generator=g).to(torch.int32)
        at = a.to(dev).transpose(1, 2).contiguous().transpose(1, 2)
        assert np.array_equal(bmm(at, b.to(dev)).cpu().numpy(), R.bmm(a.numpy(), b.numpy()))


@pytest.mark.parametrize("Z,M,K,N", [(1, 1, 64, 1), (3, 17, 193, 40), (2, 65, 127, 65), (5, 130, 321, 200),
                                     (40, 400, 64, 300), (64, 257, 128, 130), (33, 1030, 67, 70), (64, 130, 255, 140)])
def test_bmm_rows(dev, Z, M, K, N):
    """bmm where a's rows are contiguous (also at 4-byte alignment, inside a wider tensor) against rows that are not,
    b contiguous along n and along k, whole and part-filled last k steps, row and column tiles, the largest
    magnitudes."""
    from bitexact.bmm import bmm
    from bitexact.exact.consts import LIM3
    g = torch.Generator().manual_seed(Z + M + K + N)
    a = torch.randint(-LIM3, LIM3 + 1, (Z, M, K), generator=g, dtype=torch.int32)
    b = torch.randint(-LIM3, LIM3 + 1, (Z, K, N), generator=g, dtype=torch.int32)
    a[:, -1], b[:, :, -1] = LIM3, -LIM3
    ref = R.bmm(a.numpy(), b.numpy())
    wide = torch.full((Z, M, K + 5), LIM3, dtype=torch.int32)
    wide[:, :, 1:K + 1] = a
    bk = b.transpose(1, 2).contiguous().to(dev).transpose(1, 2)
    at = a.transpose(1, 2).contiguous().to(dev).transpose(1, 2)
    for x in (a.to(dev), wide.to(dev)[:, :, 1:K + 1], at):
        for y in (b.to(dev), bk):
            assert np.array_equal(bmm(x, y).cpu().numpy(), ref)


def test_bmm_int32_bound(dev):
    """The int32 limb-weight sums at the reference's bound (K < 43690): every limb -128, the largest K, and a
    mixed-sign case, against Python-int products."""
    from bitexact.bmm import bmm
    K = 43689
    x = -128 - 128 * 256 - 128 * 65536                  # three limbs of -128
    a = torch.full((1, 3, K), x, dtype=torch.long)
    b = torch.full((1, K, 5), x, dtype=torch.int32)
    got = bmm(a.to(dev), b.to(dev)).cpu().numpy()
    assert (got == x * x * K).all()
    b2 = b.clone()
    b2[0, ::2] = R.LIM3                                  # three limbs of 127
    got = bmm(a.to(dev), b2.to(dev)).cpu().numpy()
    assert (got == x * x * (K // 2) + x * R.LIM3 * ((K + 1) // 2)).all()


def test_unfused_equals_fused_attention(dev):
    """GPU bmm -> GPU softmax -> GPU bmm (the reference model's unfused order) against the fused prefill."""
    from bitexact.bmm import bmm
    from bitexact.exact import ops
    from bitexact.exact.attention import prefill
    g = torch.Generator().manual_seed(11)
    Z, gT, S, HD = 4, 96, 96, 64
    qg = torch.randint(-(1 << 22), (1 << 22) + 1, (Z, gT, HD), generator=g).to(torch.int32).to(dev)
    shg = torch.randint(-40, -10, (Z, gT, 1), generator=g).to(dev)
    K = torch.randint(-R.LIM3, R.LIM3 + 1, (Z, S, HD), generator=g).to(torch.int32).to(dev)
    V = torch.randint(-R.LIM3, R.LIM3 + 1, (Z, S, HD), generator=g).to(torch.int32).to(dev)
    qpos = (torch.arange(gT) % 24 * 4).reshape(1, gT, 1).expand(Z, gT, 1).contiguous().to(dev)
    raw = bmm(qg, K.transpose(-1, -2))
    p, den = ops.softmax(raw, qpos, shg, _lut(dev), R.L2E28)
    num = bmm(p, V)
    num2, den2 = prefill(qg, shg, K, V, qpos, _lut(dev), R.L2E28)
    assert torch.equal(num, num2) and torch.equal(den, den2)


@pytest.mark.parametrize("HD", [64, 128])
def test_int8_paged_attention(dev, HD):
    """tri_paged.attend (int8 mode) against the unfused int8 rules; M = 9 spans several 4-query tiles."""
    from bitexact.int8.consts import exp_table
    from bitexact.vllm_plugin import tri_paged
    g = torch.Generator().manual_seed(100 + HD)
    ptab = tri_paged.weight_table(exp_table(dev))
    expt = R.int8_exp_table()
    nb, bs, HKV = 64, 16, 4
    for lim, qlim in ((R.LIM3, 1 << 6), (1 << 13, 1 << 12), (1 << 10, 1 << 16)):
        c = torch.randint(-lim, lim + 1, (nb, HKV, bs, 2 * HD), generator=g).to(torch.int32)
        cl = tri_paged.to_limbs(c.to(dev))
        for Rr, M, P in [(3, 4, 600), (2, 9, 300), (6, 1, 900), (7, 4, 5)]:
            bt = torch.randint(0, nb, (Rr, 64), generator=g).to(torch.int32)
            qpos = torch.randint(0, P, (Rr, M), generator=g)
            qpos[0, 0] = -1
            q = torch.randint(-qlim, qlim + 1, (Rr, HKV, M, HD), generator=g)
            ref_num, ref_den = R.paged_attend_int8(q.numpy(), qpos.numpy(), c.numpy(), bt.numpy(), expt)
            for ns in (None, 1, 5, 64):
                num, den = tri_paged.attend(q.to(dev), qpos.to(dev), cl, bt.to(dev), ptab, nsplit=ns)
                assert np.array_equal(num.cpu().numpy(), ref_num), (Rr, M, ns, lim)
                assert np.array_equal(den.cpu().numpy(), ref_den), (Rr, M, ns, lim)


@pytest.mark.parametrize("HD,H,HKV", [(64, 32, 8), (128, 8, 2), (64, 6, 2)])
def test_rope_attend_equals_store_then_attend(dev, HD, H, HKV):
    """The decode step's fused launch (tri_exact_attn.rope_attend: RoPE, q quantization and the K / V store as the
    attention's prologue) against the two-launch path it replaces (ops.qkv_y with the cache store, then attend
    unsplit): the same num / den, the same cache bytes and the same flag; rope_attend_out (the attention output
    stage fused as well) against ops.attn_out of that num / den, one token per sequence at different
    context lengths, with a padding token (slot -1 keeps the cache unchanged) and the key at the token's own
    position read back from the slot the prologue just wrote."""
    from bitexact.exact import ops
    from bitexact.exact.consts import FT, llama3_inv_freq, rope_tables
    from bitexact.vllm_plugin import tri_exact_attn
    g = torch.Generator().manual_seed(HD + H)
    N, bs, nblk = 6, 16, 20
    cos, sin = rope_tables(400, FT, llama3_inv_freq(HD))
    cos, sin = cos.to(dev), sin.to(dev)
    W = (H + 2 * HKV) * HD
    y = torch.randint(-(1 << 30), 1 << 30, (N, W), generator=g)
    y[1, :HD] >>= 24                                   # a small q head: exponent near NEG_BIG
    pos = torch.tensor([0, 17, 100, 255, 319, 5])
    nb = 1 + N * nblk
    bt = (1 + torch.randperm(N * nblk, generator=g)).to(torch.int32).view(N, nblk)
    rmap = torch.arange(N)
    slot = bt[rmap, pos // bs].long() * bs + pos % bs
    slot[5] = -1                                       # padding: nothing stored
    c0 = torch.randint(-128, 128, (nb, HKV, bs, 8 * HD), dtype=torch.int8, generator=g).to(dev)
    lut = _lut(dev)
    l2e = R.L2E28_HD[HD]
    ca, cb = c0.clone(), c0.clone()
    fa = torch.zeros(1, dtype=torch.int32, device=dev)
    qg, shg, _, _, _ = ops.qkv_y(y.to(dev), pos.view(N, 1).to(dev), cos, sin, N, 1, (H, HKV, HD), flag=fa,
                                 store=(ca, slot.to(dev)))
    G = H // HKV
    qpos = pos.view(-1, 1).expand(-1, G).contiguous().to(dev)
    na, da = tri_exact_attn.attend(qg.view(N, HKV, G, HD), shg.view(N, HKV, G), qpos, ca, bt.to(dev), rmap.to(dev),
                                   lut, l2e, nsplit=1)
    fb = torch.zeros(1, dtype=torch.int32, device=dev)
    nb_, db = tri_exact_attn.rope_attend(y.to(dev), pos.to(dev), cos, sin, (H, HKV, HD), cb, slot.to(dev),
                                         bt.to(dev), rmap.to(dev), lut, l2e, fb)
    torch.cuda.synchronize()
    assert torch.equal(ca, cb), "cache bytes differ"
    assert torch.equal(na, nb_) and torch.equal(da, db)
    assert int(fa.item()) == int(fb.item())
    # with the attention output stage fused too: the rows ops.attn_out makes of the same num / den (twice in a
    # row: the exchange slots are left zero for the next call)
    qo, sho = ops.attn_out(na.view(N * HKV, G, HD), da.view(N * HKV, G, 1), 1, HKV)
    for _ in range(2):
        cc = c0.clone()
        fc = torch.zeros(1, dtype=torch.int32, device=dev)
        qf, shf = tri_exact_attn.rope_attend_out(y.to(dev), pos.to(dev), cos, sin, (H, HKV, HD), cc, slot.to(dev),
                                                 bt.to(dev), rmap.to(dev), lut, l2e, fc)
        torch.cuda.synchronize()
        assert torch.equal(cc, ca), "cache bytes differ (fused output stage)"
        assert torch.equal(qf, qo) and torch.equal(shf, sho)
        assert int(fc.item()) == int(fa.item())
    # the form that also writes q's limb planes (the wo linear's q_planes): the same rows, and the planes are their
    # signed base-256 digits
    cp, fp = c0.clone(), torch.zeros(1, dtype=torch.int32, device=dev)
    qp, shp, plp = tri_exact_attn.rope_attend_out(y.to(dev), pos.to(dev), cos, sin, (H, HKV, HD), cp, slot.to(dev),
                                                  bt.to(dev), rmap.to(dev), lut, l2e, fp, planes=True)
    torch.cuda.synchronize()
    assert torch.equal(cp, ca) and torch.equal(qp, qo) and torch.equal(shp, sho) and int(fp.item()) == int(fa.item())
    r = qp.long()
    for i in range(3):
        lo = ((r + 128) & 255) - 128
        assert torch.equal(plp[i].long(), lo)
        r = (r - lo) >> 8
    # a position past the rope tables flags in both forms
    pos2 = pos.clone()
    pos2[2] = 400
    fa2, fb2 = torch.zeros(1, dtype=torch.int32, device=dev), torch.zeros(1, dtype=torch.int32, device=dev)
    ops.qkv_y(y.to(dev), pos2.view(N, 1).to(dev), cos, sin, N, 1, (H, HKV, HD), flag=fa2, store=(c0.clone(),
                                                                                                     slot.to(dev)))
    tri_exact_attn.rope_attend(y.to(dev), pos2.to(dev), cos, sin, (H, HKV, HD), c0.clone(), slot.to(dev), bt.to(dev),
                               rmap.to(dev), lut, l2e, fb2)
    assert int(fa2.item()) == 1 and int(fb2.item()) == 1
