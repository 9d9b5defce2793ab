"""HIP row stages against the reference's own vectors (tests/golden/reference_vectors.npz) and the oracle:
RMSNorm + quantization (segs.norm_quant), masked softmax weights (segs.softmax), attention output rule."""

import os

import numpy as np
import pytest
import torch

from oracle import bxref as R

pytestmark = pytest.mark.gpu

GOLD = np.load(os.path.join(os.path.dirname(__file__), "golden", "reference_vectors.npz"))


@pytest.mark.parametrize("D", [512, 2048, 4096])
def test_norm_quant_golden(dev, D):
    from bitexact.exact import ops
    x = torch.from_numpy(GOLD[f"rms{D}_x"]).to(dev)
    q, sh, err = ops.norm_quant(x, torch.from_numpy(GOLD[f"nq{D}_gm"]).to(dev), torch.from_numpy(GOLD[f"nq{D}_ge"]).to(dev))
    assert np.array_equal(q.cpu().numpy(), GOLD[f"nq{D}_q"]) and np.array_equal(sh.cpu().numpy(), GOLD[f"nq{D}_sh"])
    assert bool(err) == bool(GOLD[f"nq{D}_err"])


def test_norm_quant_random(dev):
    from bitexact.exact import ops
    g = torch.Generator().manual_seed(2)
    for M in (1, 37):
        x = torch.randint(-(1 << 30), 1 << 30, (M, 2048), generator=g)
        x = x >> torch.randint(0, 24, (M, 1), generator=g)
        gm = torch.randint(-255, 256, (2048,), generator=g)
        ge = torch.randint(-14, -6, (2048,), generator=g)
        q, sh, err = ops.norm_quant(x.to(dev), gm.to(dev), ge.to(dev))
        rq, rsh, rerr = R.norm_quant(x.numpy(), gm.numpy(), ge.numpy())
        assert np.array_equal(q.cpu().numpy(), rq) and np.array_equal(sh.cpu().numpy(), rsh) and bool(err) == rerr
    x = torch.zeros(2, 512, dtype=torch.long)
    x[1, 3] = 1 << 41                                          # bound violation sets the flag
    _, _, err = ops.norm_quant(x.to(dev), torch.ones(512, dtype=torch.long, device=dev),
                               torch.full((512,), -7, dtype=torch.long, device=dev))
    assert bool(err)


@pytest.mark.parametrize("many", [False, True])
@pytest.mark.parametrize("D", [2, 64, 1024, 2048, 4096])
@pytest.mark.parametrize("big", [False, True])
def test_norm_row_forms(dev, many, D, big):
    """RMSNorm at both block sizes (few rows; two per CU) and its row widths, against the oracle on the edge rows and
    between 16-byte and single-element accesses (rows of odd stride) on all: N(0, 1) rows, a zero row, a row of one
    value, values next to 2^40, and with `big` what float64 does not hold (a value of 2^52, one of 2^60, gamma
    exponents that take quotients past 2^50), where the int64 rule runs; q's limb planes against q."""
    from bitexact.exact import ops
    M = (2 * torch.cuda.get_device_properties(dev).multi_processor_count if many else 0) + 9
    g = torch.Generator().manual_seed(D + M)
    x = (torch.randn(M, D, generator=g) * 2.0 ** 24).long()
    x[1], x[2], x[2, D // 2] = 0, 0, -1
    x[3] = torch.randint(-(1 << 40) + 1, 1 << 40, (D,), generator=g)
    x[4] >>= 20
    gm = torch.randint(-255, 256, (D,), generator=g)
    ge = torch.randint(-14, -6, (D,), generator=g)
    if big:
        x[5, 0], x[6, D - 1] = 1 << 52, -(1 << 60)
        ge[D - 1] = 11
    rows = [0, 1, 2, 3, 4, 5, 6, 7, M - 1]
    xd, gd, ed = x.to(dev), gm.to(dev), ge.to(dev)
    q, sh, err = ops.norm_quant(xd, gd, ed)
    rq, rsh, rerr = R.norm_quant(x[rows].numpy(), gm.numpy(), ge.numpy())
    assert np.array_equal(q[rows].cpu().numpy(), rq) and np.array_equal(sh[rows].cpu().numpy(), rsh) and bool(err) == rerr
    odd = torch.zeros(M, D + 1, dtype=torch.long, device=dev)
    odd[:, :D] = xd
    q2, sh2, _ = ops.norm_quant(odd[:, :D], gd, ed)
    assert torch.equal(q, q2) and torch.equal(sh, sh2)
    y = torch.randint(-(1 << 24), 1 << 24, (M, D), generator=g)
    ids = torch.randint(0, M, (M,), generator=g)
    emb = (x >> 20).to(torch.int32)
    for planes in ([False, True] if D % 16 == 0 else [False]):
        xo, qa, sha, _ = ops.add_norm_y(y.to(dev), (x - y).to(dev), gd, ed, planes=planes)
        qa, pl = qa if planes else (qa, None)
        assert torch.equal(xo, xd) and torch.equal(qa, q) and torch.equal(sha, sh)
        if planes:
            p = pl.long()
            assert torch.equal(p[0] + 256 * p[1] + 65536 * p[2], q.long())
    xe, qe, she, _ = ops.embed_norm(emb.to(dev), ids.to(dev), gd, ed)
    re = emb[ids].long()
    rq, rsh, _ = R.norm_quant(re[rows].numpy(), gm.numpy(), ge.numpy())
    assert torch.equal(xe.cpu(), re) and np.array_equal(qe[rows].cpu().numpy(), rq)
    assert np.array_equal(she[rows].cpu().numpy(), rsh)


@pytest.mark.parametrize("T", [5, 517])
@pytest.mark.parametrize("hkv,grp,HD", [(8, 4, 64), (8, 4, 128), (2, 3, 64)])
def test_attn_out_row_forms(dev, T, hkv, grp, HD):
    """The attention output stage at both block sizes and widths against the oracle: averages of values (den 2^22 ..
    2^34), exact halves, rows that see no key (den 0), rows float64 does not hold (num of 2^59, den of 2^35); and the
    LDS form (num rows of odd stride) on the same rows."""
    from bitexact.exact import ops
    g = torch.Generator().manual_seed(T + HD)
    shape = (hkv, grp * T, HD)
    den = torch.randint(1 << 22, 1 << 30, (*shape[:2], 1), generator=g)
    num = (den.double() * torch.randn(shape, generator=g).double() * 2.0 ** 19).long()
    num[:, 1] = den[:, 1] // 64 * torch.randint(-99, 100, (hkv, HD), generator=g)      # num 2^5 / den near halves
    den[:, 2] = 0
    num[0, 3, 5] = 1 << 59
    den[1, 4], den[0, 0] = 1 << 35, (1 << 34) - 1
    q, sh = ops.attn_out(num.to(dev), den.to(dev), T, hkv)
    odd = torch.zeros(hkv, grp * T, HD + 1, dtype=torch.long, device=dev)
    odd[..., :HD] = num.to(dev)
    q2, sh2 = ops.attn_out(odd[..., :HD], den.to(dev), T, hkv)
    assert torch.equal(q, q2) and torch.equal(sh, sh2)
    o = np.where(den.numpy() > 0, R.attn_div(num.numpy(), np.maximum(den.numpy(), 1)), 0)
    o = o.reshape(1, hkv, grp, T, HD).transpose(0, 3, 1, 2, 4).reshape(T, hkv * grp * HD)
    keep = [r for r in range(T) if r != 4]                          # (den 2^35 is past the rule's 2^34)
    rq, rsh = R.quant(o, -R.FR)
    assert np.array_equal(q.cpu().numpy()[keep], rq[keep]) and np.array_equal(sh.cpu().numpy()[keep], rsh[keep])


@pytest.mark.parametrize("hd", [64, 128])
def test_softmax_golden(dev, hd):
    from bitexact.exact import ops
    raw = torch.from_numpy(GOLD[f"sm{hd}_raw"]).to(dev)
    qpos = torch.from_numpy(GOLD[f"sm{hd}_qpos"]).to(dev)
    sh = torch.from_numpy(GOLD[f"sm{hd}_sh"]).to(dev)
    lut = torch.from_numpy(R.exp2_table()).to(dev)
    p, den = ops.softmax(raw, qpos, sh, lut, R.L2E28_HD[hd])
    assert np.array_equal(p.cpu().numpy().astype(np.int64), GOLD[f"sm{hd}_p"])
    assert np.array_equal(den.cpu().numpy(), GOLD[f"sm{hd}_den"])


def test_attn_out(dev):
    from bitexact.exact import ops
    g = torch.Generator().manual_seed(5)
    B, HKV, grp, T, HD = 2, 8, 4, 9, 64
    Z = B * HKV
    num = torch.randint(-(1 << 60), 1 << 60, (Z, grp * T, HD), generator=g)
    den = torch.randint(1 << 22, 1 << 34, (Z, grp * T, 1), generator=g)
    q, sh = ops.attn_out(num.to(dev), den.to(dev), T, HKV)
    o = R.attn_div(num.numpy(), den.numpy())
    o = o.reshape(B, HKV, grp, T, HD).transpose(0, 3, 1, 2, 4).reshape(B * T, HKV * grp * HD)
    rq, rsh = R.quant(o, -R.FR)
    assert np.array_equal(q.cpu().numpy(), rq) and np.array_equal(sh.cpu().numpy(), rsh)
