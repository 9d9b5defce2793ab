"""The work whose speed is followed from one version to the next: the exact and int8 linears, the integer attentions,
the row stages, bmm and the whole exact engine, each through its public entry point, over the sizes of
Llama-3.2-1B (D 2048, 32 / 8 heads of 64, FF 8192, V 128256) and of a generic 4096-wide model with heads of 128.

Every output is an integer fixed by the integer rules, so every tolerance is "exact"."""

import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "bitexact-llm_amd"))

FR, FN, FV = 24, 40, 19
L2E = {64: 387270501, 128: 273841598}
# (N, K) of the linears: qkv, o, gate|up, down at D 2048, and qkv, o at D 4096
WIDTHS = [(3072, 2048), (2048, 2048), (16384, 2048), (2048, 8192), (6144, 4096), (4096, 4096)]
H, HKV = 32, 8


def listed():
    return [
        # one token of one sequence through one linear: the smallest call, all latency
        {"name": "linear_1x3072x2048", "kind": "linear", "M": 1, "N": 3072, "K": 2048},
        # a ragged prompt through the down projection
        {"name": "linear_777x2048x8192", "kind": "linear", "M": 777, "N": 2048, "K": 8192},
        # a full prefill chunk through the fused gate|up
        {"name": "linear_2048x16384x2048", "kind": "linear", "M": 2048, "N": 16384, "K": 2048},
        # int8 mode: a decode step's linears, 8 layers deep, replayed from the graph a serving loop keeps
        {"name": "int8_decode_8", "kind": "int8_decode", "M": 8, "nl": 2, "layers": 8},
        # int8 mode: a prefill chunk through the fused gate|up
        {"name": "int8_2048x16384x2048", "kind": "int8", "M": 2048, "N": 16384, "K": 2048, "nl": 2},
        # causal attention of a prompt batch over the contiguous cache
        {"name": "attn_prefill_4x1024_hd64", "kind": "attn_prefill", "B": 4, "T": 1024, "HD": 64},
        # one ragged prompt, heads of 128
        {"name": "attn_prefill_1x1337_hd128", "kind": "attn_prefill", "B": 1, "T": 1337, "HD": 128},
        # a decode batch over long paged contexts
        {"name": "attn_paged_16x4096_hd64", "kind": "attn_paged", "B": 16, "ctx": 4096, "HD": 64, "mode": "exact"},
        # the row stages of one layer over a prompt batch
        {"name": "stages_4096", "kind": "stages", "M": 4096, "D": 2048, "FF": 8192, "HD": 64},
        # the unfused attention's weights times values
        {"name": "bmm_pv_16x4096x1024x64", "kind": "bmm", "Z": 16, "M": 4096, "K": 1024, "N": 64, "side": "pv"},
        # the whole model, one greedy decode step at batch 32 (the step's graph, as a serving loop keeps it)
        {"name": "engine_decode_32x1024", "kind": "engine_decode", "B": 32, "ctx": 1024},
        # the whole model, prefill of 8 prompts of 512 into the paged cache
        {"name": "engine_prefill_8x512", "kind": "engine_prefill", "B": 8, "T": 512},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "int8", "int8", "int8_decode", "attn_prefill", "attn_prefill", "attn_paged",
                       "attn_paged", "stages", "bmm", "engine_decode", "engine_prefill"])
    if kind in ("linear", "int8"):
        N, K = rng.choice(WIDTHS)
        if rng.random() < 0.3:
            N -= rng.randrange(1, 64)                      # ragged widths (a vocabulary slice, a shard)
        c = {"kind": kind, "M": _log_int(rng, 1, 2048), "N": N, "K": K}
        if kind == "int8":
            c["nl"] = rng.choice([1, 2, 2, 3])
        return c
    if kind == "int8_decode":
        return {"kind": kind, "M": _log_int(rng, 1, 64), "nl": rng.choice([1, 2, 2]), "layers": rng.randrange(4, 9)}
    if kind == "attn_prefill":
        B = rng.choice([1, 2, 3, 4])
        return {"kind": kind, "B": B, "T": _log_int(rng, 48, 1500 // B + 400), "HD": rng.choice([64, 64, 128])}
    if kind == "attn_paged":
        B = _log_int(rng, 1, 64)
        return {"kind": kind, "B": B, "ctx": _log_int(rng, 64, min(4096, 65536 // B)), "HD": rng.choice([64, 64, 128]),
                "mode": rng.choice(["exact", "exact", "int8"])}
    if kind == "stages":
        D, FF, HD = rng.choice([(2048, 8192, 64), (4096, 14336, 128)])
        return {"kind": kind, "M": _log_int(rng, 1, 4096 if D == 2048 else 2048), "D": D, "FF": FF, "HD": HD}
    if kind == "bmm":
        HD, S = rng.choice([64, 128]), _log_int(rng, 64, 2000)
        c = {"kind": kind, "Z": rng.choice([8, 16]), "M": 4 * _log_int(rng, 16, 1024), "side": rng.choice(["pv", "qk"])}
        return {**c, "K": S, "N": HD} if c["side"] == "pv" else {**c, "K": HD, "N": S}
    if kind == "engine_decode":
        return {"kind": kind, "B": _log_int(rng, 1, 48), "ctx": _log_int(rng, 64, 1400)}
    B = rng.randrange(1, 7)
    return {"kind": kind, "B": B, "T": _log_int(rng, 32, 3000 // B)}


# ---- inputs ----
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(g, *shape, bits=FR):
    """N(0, 1) at `bits` fractional bits, int64 (a residual stream, a linear's output)."""
    return (torch.randn(*shape, generator=g, device="cuda") * 2.0 ** bits).long()


def _bf16_weight(g, n, k):
    return (torch.randn(n, k, generator=g, device="cuda") * 0.02).to(torch.bfloat16)


def _activation_rows(g, M, K):
    """Quantized activation rows q int32 [M, K], |q| <= 2^22, with their exponents: value q 2^sh ~ N(0, 1)."""
    x = torch.randn(M, K, generator=g, device="cuda", dtype=torch.float64)
    e = torch.frexp(x.abs().amax(-1)).exponent.long()
    q = torch.floor(torch.ldexp(x, (22 - e)[:, None]) + 0.5).to(torch.int32)
    return q, e - 22


def _limb_rows(g, M, K, nl):
    """int8 mode's stacked limb rows [nl M, K] of N(0, 1) rows quantized to nl limbs."""
    x = torch.randn(M, K, generator=g, device="cuda", dtype=torch.float64)
    lim = {1: 127, 2: 32512, 3: 8323072}[nl]
    q = torch.round(x * (lim / x.abs().amax(-1, keepdim=True))).long()
    out = []
    for _ in range(nl):
        lo = ((q + 128) & 255) - 128
        out.append(lo)
        q = (q - lo) >> 8
    return torch.cat(out).to(torch.int8)


def _int8_weight(g, n, k):
    return torch.randint(-127, 128, (n, k), generator=g, device="cuda", dtype=torch.int8)


def _rope(HD, n=4096):
    from bitexact.exact.consts import FT, llama3_inv_freq, rope_tables
    return tuple(t.cuda() for t in rope_tables(n, FT, llama3_inv_freq(HD)))


def _heads(g, B, T, HD):
    """Rotated, quantized queries and integer K / V of B prompts of T tokens (what the qkv linear's output gives)."""
    from bitexact.exact import ops
    y = _normal(g, B * T, (H + 2 * HKV) * HD)
    pos = torch.arange(T, device="cuda").repeat(B, 1)
    cos, sin = _rope(HD)
    qg, shg, k, v, _ = ops.qkv_y(y, pos, cos, sin, B, T, (H, HKV, HD))
    return qg, shg, k, v, pos


def _fill(g, cache, blocks):
    """K ~ N(0, 1) at 17 bits and V at 19 in every slot of the cache's blocks 1.."""
    from bitexact.vllm_plugin import tri_paged
    _, hkv, bs, w = cache.shape
    hd, per = w // 8, 1024
    for b0 in range(1, blocks, per):
        b1 = min(blocks, b0 + per)
        slot = torch.arange(b0 * bs, b1 * bs, device="cuda")
        k = (torch.randn(slot.numel(), hkv, hd, generator=g, device="cuda") * 2.0 ** 17).to(torch.int32)
        v = (torch.randn(slot.numel(), hkv, hd, generator=g, device="cuda") * 2.0 ** 19).to(torch.int32)
        tri_paged.store(cache, slot, k, v)


def _graph(step):
    """`step` captured once, as a serving loop keeps its decode step."""
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        out = step()
    torch.cuda.synchronize()
    return graph, out


DECODE_LINEARS = [(3072, 2048), (2048, 2048), (16384, 2048), (2048, 8192)]


def prepare(case, seed):
    from bitexact.exact import consts
    kind, g = case["kind"], _gen(seed)
    s = dict(case)
    if kind == "linear":
        from bitexact.vllm_plugin.exact_gemm import FusedLin
        from bitexact.exact.model import Lin
        dec = consts.decompose(_bf16_weight(g, case["N"], case["K"]))
        s["lin"] = FusedLin(Lin({f"w.{k}": v for k, v in dec.items()}, "w", "cuda"))
        s["q"], s["sh"] = _activation_rows(g, case["M"], case["K"])
        s["flag"] = torch.zeros(1, dtype=torch.int32, device="cuda")
    elif kind == "int8":
        s["w"] = _int8_weight(g, case["N"], case["K"])
        s["a"] = _limb_rows(g, case["M"], case["K"], case["nl"])
    elif kind == "int8_decode":
        from bitexact.int8.gemm_skinny import int_mm_join
        ws = [[_int8_weight(g, n, k) for n, k in DECODE_LINEARS] for _ in range(case["layers"])]
        rows = {k: _limb_rows(g, case["M"], k, case["nl"]) for k in (2048, 8192)}
        s["w"], s["rows"] = ws, rows
        s["graph"], s["y"] = _graph(lambda: [int_mm_join(rows[w.shape[1]], w, case["M"], case["nl"])
                                             for layer in ws for w in layer])
    elif kind == "attn_prefill":
        B, T, HD = case["B"], case["T"], case["HD"]
        s["qg"], s["shg"], k, v, pos = _heads(g, B, T, HD)
        s["K"], s["V"] = (t.permute(0, 2, 1, 3).reshape(B * HKV, T, HD).to(torch.int32) for t in (k, v))
        s["qpos"] = pos[:, None, None, :].expand(B, HKV, H // HKV, T).reshape(B * HKV, -1, 1)
        s["lut"] = consts.exp2_table("cuda")
    elif kind == "attn_paged":
        B, HD, bs = case["B"], case["HD"], 16
        nblk = -(-case["ctx"] // bs)
        s["cache"] = torch.zeros(1 + B * nblk, HKV, bs, 8 * HD, dtype=torch.int8, device="cuda")
        _fill(g, s["cache"], 1 + B * nblk)
        s["bt"] = (1 + torch.randperm(B * nblk, generator=g, device="cuda")).to(torch.int32).view(B, nblk)
        G = H // HKV
        s["qpos"] = torch.full((B, G), case["ctx"] - 1, dtype=torch.long, device="cuda")
        if case["mode"] == "int8":
            from bitexact.int8.consts import exp_table
            from bitexact.vllm_plugin.tri_paged import weight_table
            s["q"] = _normal(g, B, HKV, G, HD, bits=14)
            s["ptab"] = weight_table(exp_table("cuda"))
        else:
            y = _normal(g, B, (H + 2 * HKV) * HD)
            from bitexact.exact import ops
            pos = torch.full((B, 1), case["ctx"] - 1, dtype=torch.long, device="cuda")
            qg, shg, _, _, _ = ops.qkv_y(y, pos, *_rope(HD), B, 1, (H, HKV, HD))
            s["q"], s["sh"] = qg.view(B, HKV, G, HD), shg.view(B, HKV, G)
            s["rmap"], s["lut"] = torch.arange(B, device="cuda"), consts.exp2_table("cuda")
    elif kind == "stages":
        M, D, FF, HD = case["M"], case["D"], case["FF"], case["HD"]
        s["emb"] = (torch.randn(32000, D, generator=g, device="cuda") * 0.02 * 2.0 ** FR).to(torch.int32)
        s["ids"] = torch.randint(0, 32000, (M,), generator=g, device="cuda")
        one = torch.ones(D, device="cuda") + 0.1 * torch.randn(D, generator=g, device="cuda")
        s["gamma"] = consts.bf16_parts(one.to(torch.bfloat16))
        s["y_qkv"] = _normal(g, M, (H + 2 * HKV) * HD)
        s["pos"] = torch.arange(M, device="cuda").remainder(4096).view(1, M)
        s["cos"], s["sin"] = _rope(HD)
        s["den"] = torch.randint(1 << 22, 1 << 30, (HKV, M * (H // HKV), 1), generator=g, device="cuda")
        s["num"] = (s["den"].double() * torch.randn(HKV, M * (H // HKV), HD, generator=g, device="cuda").double()
                    * 2.0 ** FV).long()
        s["y_o"], s["gu"] = _normal(g, M, D), _normal(g, M, 2 * FF)
        s["lut"] = consts.exp2_table("cuda")
        s["flag"] = torch.zeros(1, dtype=torch.int32, device="cuda")
    elif kind == "bmm":
        Z, M, N, K = case["Z"], case["M"], case["N"], case["K"]
        if case["side"] == "pv":                           # weights in [0, 2^22], values at 19 bits
            s["a"] = torch.randint(0, (1 << 22) + 1, (Z, M, K), generator=g, device="cuda", dtype=torch.int32)
            s["b"] = _normal(g, Z, K, N, bits=FV).to(torch.int32)
        else:                                              # quantized queries, keys transposed in memory
            s["a"] = _activation_rows(g, Z * M, K)[0].view(Z, M, K)
            s["b"] = _normal(g, Z, N, K, bits=17).to(torch.int32).transpose(1, 2)
    else:
        from bitexact.vllm_plugin.exact_run import ExactEngine
        eng = ExactEngine(consts.random_constants(None, seed=seed, device="cuda"), "cuda")
        B, bs = case["B"], 16
        last = case["ctx"] if kind == "engine_decode" else case["T"] - 1
        nblk = last // bs + 1
        kvs = eng.new_cache(1 + B * nblk, bs)
        bt = (1 + torch.randperm(B * nblk, generator=g, device="cuda")).to(torch.int32).view(B, nblk)
        if kind == "engine_decode":
            for c in kvs:
                _fill(g, c, 1 + B * nblk)
            pos = torch.full((B,), last, dtype=torch.long, device="cuda")
            rmap = torch.arange(B, device="cuda")
        else:
            pos = torch.arange(case["T"], device="cuda").repeat(B)
            rmap = torch.arange(B, device="cuda").repeat_interleave(case["T"])
        ids = torch.randint(0, eng.V, (pos.numel(),), generator=g, device="cuda")
        slot = bt[rmap, pos // bs].long() * bs + pos % bs
        s.update(eng=eng, kvs=kvs, bt=bt, pos=pos, rmap=rmap, ids=ids, slot=slot)
        if kind == "engine_decode":
            def step():
                x = eng.forward(kvs, ids, pos, slot, bt, rmap, one_per_seq=True)
                logits = eng.logits(x)
                return x, logits, eng.greedy(logits)
            s["graph"], s["y"] = _graph(step)
    return s


# ---- one pass ----
def run(s):
    kind = s["kind"]
    if kind == "linear":
        return s["lin"](s["q"], s["sh"], s["flag"])
    if kind == "int8":
        from bitexact.int8.gemm_skinny import int_mm_join
        return int_mm_join(s["a"], s["w"], s["M"], s["nl"])
    if kind in ("int8_decode", "engine_decode"):
        s["graph"].replay()
        return s["y"]
    if kind == "attn_prefill":
        from bitexact.exact.attention import prefill
        return prefill(s["qg"], s["shg"], s["K"], s["V"], s["qpos"], s["lut"], L2E[s["HD"]])
    if kind == "attn_paged":
        from bitexact.vllm_plugin import tri_exact_attn, tri_paged
        if s["mode"] == "int8":
            return tri_paged.attend(s["q"], s["qpos"], s["cache"], s["bt"], s["ptab"])
        return tri_exact_attn.attend(s["q"], s["sh"], s["qpos"], s["cache"], s["bt"], s["rmap"], s["lut"], L2E[s["HD"]])
    if kind == "stages":
        from bitexact.exact import ops
        fl, M = s["flag"], s["M"]
        x, q0, sh0, _ = ops.embed_norm(s["emb"], s["ids"], *s["gamma"], flag=fl)
        qg, shg, k, v, _ = ops.qkv_y(s["y_qkv"], s["pos"], s["cos"], s["sin"], 1, M, (H, HKV, s["HD"]), flag=fl)
        qo, sho = ops.attn_out(s["num"], s["den"], M, HKV)
        x, q1, sh1, _ = ops.add_norm_y(s["y_o"], x, *s["gamma"], flag=fl)
        q2, sh2, _ = ops.gu_silu_y(s["gu"], s["lut"], flag=fl)
        return [x, q0, sh0, qg, shg, k, v, qo, sho, q1, sh1, q2, sh2]
    if kind == "bmm":
        from bitexact.bmm import bmm
        return bmm(s["a"], s["b"])
    eng = s["eng"]
    x = eng.forward(s["kvs"], s["ids"], s["pos"], s["slot"], s["bt"], s["rmap"])
    logits = eng.logits(x.view(s["B"], s["T"], -1)[:, -1].contiguous())
    return [x, logits] + s["kvs"]


def _layer_ops():
    return sum(n * k for n, k in DECODE_LINEARS)


def work(case):
    """What a pass cannot do without: bytes of each input and output once, int8 multiply-adds of the limb products
    (9 of 3 x 3 limbs; nl in int8 mode) times two."""
    c, kind = case, case["kind"]
    if kind == "linear":
        M, N, K = c["M"], c["N"], c["K"]
        return {"bytes": 3 * N * K + 4 * M * K + 8 * M * N + 16 * N + 8 * M, "flops": 18 * M * N * K}
    if kind == "int8":
        M, N, K, nl = c["M"], c["N"], c["K"], c["nl"]
        return {"bytes": N * K + nl * M * K + 8 * M * N, "flops": 2 * nl * M * N * K}
    if kind == "int8_decode":
        M, nl = c["M"], c["nl"]
        return {"bytes": c["layers"] * sum(n * k + nl * M * k + 8 * M * n for n, k in DECODE_LINEARS),
                "flops": c["layers"] * 2 * nl * M * _layer_ops()}
    if kind == "attn_prefill":
        B, T, HD = c["B"], c["T"], c["HD"]
        return {"bytes": B * T * (H * (4 * HD + 8 + 8) + 2 * HKV * 4 * HD + H * (8 * HD + 8)),
                "flops": 2 * 18 * HD * B * H * T * (T + 1) // 2}
    if kind == "attn_paged":
        B, S, HD = c["B"], c["ctx"], c["HD"]
        return {"bytes": B * (HKV * S * 6 * HD + H * (4 * HD + 8 * HD + 16)), "flops": 2 * 18 * HD * B * H * S}
    if kind == "stages":
        M, D, FF, HD = c["M"], c["D"], c["FF"], c["HD"]
        # embed + norm; rope + grouping; attention output; add + norm; gate|up
        b = (4 + 8 + 4) * D + (8 * (H + 2 * HKV) + 4 * H + 16 * HKV) * HD + (8 + 4) * H * HD
        return {"bytes": M * (b + (8 + 8 + 8 + 4) * D + (16 + 4) * FF), "flops": 0}
    if kind == "bmm":
        Z, M, N, K = c["Z"], c["M"], c["N"], c["K"]
        return {"bytes": Z * (4 * M * K + 4 * K * N + 8 * M * N), "flops": 18 * Z * M * N * K}
    L, V, D = 16, 128256, 2048
    if kind == "engine_decode":
        B, S = c["B"], c["ctx"] + 1
        return {"bytes": 3 * (L * _layer_ops() + V * D) + L * B * S * HKV * 6 * 64 + 8 * B * (V + D),
                "flops": 18 * B * (L * _layer_ops() + V * D) + L * 36 * 64 * B * H * S}
    B, T = c["B"], c["T"]
    return {"bytes": 3 * (L * _layer_ops() + V * D) + L * B * T * HKV * 6 * 64 + 8 * B * (V + T * D),
            "flops": 18 * (B * T * L * _layer_ops() + B * V * D) + L * 36 * 64 * B * H * T * (T + 1) // 2}


def tolerance(case):
    return "exact"


def exact(case, seed):
    """The matrix products of the linears and of bmm in plain torch, 64 bits; the other stages' integers have no plain
    floating counterpart."""
    kind, g = case["kind"], _gen(seed)
    if kind == "linear":
        w = _bf16_weight(g, case["N"], case["K"]).double()
        q, sh = _activation_rows(g, case["M"], case["K"])
        return torch.floor(torch.ldexp(q.double() @ w.t().contiguous(), (sh + FR)[:, None]) + 0.5).long()
    if kind == "int8":
        w = _int8_weight(g, case["N"], case["K"]).double().t().contiguous()
        rows = _limb_rows(g, case["M"], case["K"], case["nl"]).double().view(case["nl"], case["M"], case["K"])
        return sum((rows[i] @ w).long() << (8 * i) for i in range(case["nl"]))
    if kind == "bmm":
        s = prepare(case, seed)
        a, b = s["a"].long(), s["b"].contiguous().double()
        lo = a & 4095
        return (lo.double() @ b).long() + (((a - lo) >> 12).double() @ b).long() * 4096
    return None
