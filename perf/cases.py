"""Performance cases of the selected-quant decode framework: what a serving or
research program has it do, through its public entry points.

``listed()`` holds the fixed cases, ``draw(rng)`` one more case of the same
ranges. ``prepare(case, seed)`` makes what the program has in hand before the
call, ``run(state)`` is one pass, ``exact(case, seed)`` the same outputs from
plain torch in 64 bits. The kinds:

  decode       selected-page mixed-precision decode, both reference-shaped APIs
  mla_paged    MLA latent decode over paged latent pools (the serving form)
  mla_api      MLA decode over a 1-D page table, with the output projection
  dense        dense softmax attention (prefill and decode shapes)
  blocks       semantic-block attention over a layout's selected tokens
  iqa          attention over fake-quantised selected blocks
  quantize     quantise-on-write of float16 pages into the four pools
  tables       page tables from routing decisions
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "intent-attention-kernel_amd"))

import intent_attention as ia  # noqa: E402
from intent_attention.intent_quant_decode import IntentQuantKernelConfig, intent_quant_decode_attention_triton  # noqa: E402

PS = 16                                       # tokens per page
FP16, INT8, SKIP, FP8, INT4, INT4R = range(6)  # the decode's native page tags
_NAME = {FP16: "fp16", INT8: "int8", FP8: "fp8", INT4: "int4", INT4R: "int4r"}
_DTYPE = {"float16": torch.float16, "bfloat16": torch.bfloat16, "float32": torch.float32}
_SIZE = {"float16": 2, "bfloat16": 2, "float32": 4}
# page precision mixes, as tag: share
_MIX = {
    "fp16_int8": {FP16: .5, INT8: .5},                       # the two precisions of the reference's pools
    "four": {FP16: .25, FP8: .25, INT8: .30, INT4: .20},     # the headline mix
    "residual": {FP16: .10, INT8: .30, INT4R: .60},
    "fp16": {FP16: 1.0},
    "skips": {FP16: .3, INT8: .5, SKIP: .2},
}


def listed():
    return [
        # the smallest step: one sequence, 32 selected pages of 16 tokens, 8 heads of 64 (launches and latency)
        dict(name="decode_small", kind="decode", api="fused", B=1, Hq=8, Hkv=8, D=64, W=32, share=0.5,
             mix="fp16_int8", q="float16", ragged=False),
        # an ordinary ragged batch through the second API: float32 queries, odd counts, GQA of five
        dict(name="decode_ragged_f32", kind="decode", api="sibling", B=5, Hq=20, Hkv=4, D=64, W=151, share=0.5,
             mix="skips", q="float32", ragged=True),
        # four 128k-token sequences, 15 % of the pages, mostly two-scale residual INT4
        dict(name="decode_residual_128k", kind="decode", api="fused", B=4, Hq=32, Hkv=8, D=128, W=1228, share=0.15,
             mix="residual", q="float16", ragged=False),
        # the headline step: 32 sequences of 64k tokens, 40 % of the pages, four precisions
        dict(name="decode_mixed_64k", kind="decode", api="fused", B=32, Hq=32, Hkv=8, D=128, W=1638, share=0.4,
             mix="four", q="float16", ragged=False),
        # latent decode of a whole 128-head model, half the pages of 16k tokens, FP8 / INT8 latents
        dict(name="mla_serving", kind="mla_paged", B=32, H=128, dqk=576, dv=512, W=512, pool="codes", q="float16",
             ragged=False),
        # the same model's heads shared over eight GPUs: 16 heads here, float16 latents, ragged lengths
        dict(name="mla_head_shard", kind="mla_paged", B=8, H=16, dqk=576, dv=512, W=301, pool="fp16", q="bfloat16",
             ragged=True),
        # the reference's MLA decode API with its projection: 32 queries over 8,192 selected latent rows
        dict(name="mla_projected", kind="mla_api", B=32, q_len=1, T=16384, page=64, pages=128, dc=576, d_out=4096,
             q="float32", c="float16"),
        # causal prefill of a 2k-token prompt, 32 heads of 128
        dict(name="prefill_f16", kind="dense", heads=32, tq=2048, tk=2048, D=128, dtype="float16", causal=True,
             mask=False),
        # 128 queries over the selected blocks of a 4k context in float32 (the reference's published comparison)
        dict(name="blocks_f32", kind="blocks", heads=8, tq=128, tk=4096, D=64, nblocks=16, dtype="float32",
             causal=False),
        # attention over three fake-quantised quarter-context blocks, 8 queries of 32 heads
        dict(name="intent_quant_f32", kind="iqa", heads=32, tq=8, tk=4096, D=128, nblocks=4,
             precs="INT8,INT4_RESIDUAL,FP8"),
        # one write of fresh pages into each of the four quantised pools
        dict(name="quantize_pages", kind="quantize", pages=32771, D=128),
        # the routing decisions of 32 sequences turned into kernel page tables
        dict(name="page_tables", kind="tables", B=32, H=8, T=65536, share=0.4),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "mla_paged", "mla_paged", "mla_api", "dense", "dense",
                       "blocks", "iqa", "quantize", "tables"])
    if kind == "decode":
        Hq, Hkv = rng.choice([(8, 8), (16, 4), (20, 4), (32, 8), (28, 4), (12, 6), (32, 2)])
        B = _log(rng, 1, 32)
        return dict(kind=kind, api=rng.choice(["fused", "sibling"]), B=B, Hq=Hq, Hkv=Hkv, D=rng.choice([64, 128]),
                    W=_log(rng, 8, min(1638, 400000 // (B * Hkv))), share=0.4, mix=rng.choice(sorted(_MIX)),
                    q=rng.choice(["float16", "bfloat16", "float32"]), ragged=rng.random() < 0.6)
    if kind == "mla_paged":
        dqk, dv = rng.choice([(576, 512), (576, 512), (512, 512), (128, 128)])
        return dict(kind=kind, B=_log(rng, 1, 32), H=rng.choice([8, 16, 16, 24, 32, 64, 128]), dqk=dqk, dv=dv,
                    W=_log(rng, 8, 512), pool=rng.choice(["codes", "fp16", "mixed"]),
                    q=rng.choice(["float16", "bfloat16", "float32"]), ragged=rng.random() < 0.6)
    if kind == "mla_api":
        T = _log(rng, 512, 16384)
        page = rng.choice([16, 64])
        return dict(kind=kind, B=_log(rng, 1, 32), q_len=rng.choice([1, 1, 2, 3]), T=T, page=page,
                    pages=max(1, min(T // page, _log(rng, 4, 8192 // page))), dc=rng.choice([128, 512, 576]),
                    d_out=rng.choice([1024, 4096]), q=rng.choice(["float32", "float16", "bfloat16"]),
                    c=rng.choice(["float32", "float16", "bfloat16"]))
    if kind == "dense":
        tq = rng.choice([1, _log(rng, 2, 64), _log(rng, 64, 2048), _log(rng, 64, 2048)])
        tk = _log(rng, max(tq, 32), 4096 if tq == 1 else max(2048, tq))
        return dict(kind=kind, heads=_log(rng, 2, 16), tq=tq, tk=tk, D=rng.choice([64, 80, 96, 128, 192]),
                    dtype=rng.choice(["float16", "bfloat16", "float32"]), causal=rng.random() < 0.5,
                    mask=rng.random() < 0.25)
    if kind == "blocks":
        return dict(kind=kind, heads=_log(rng, 2, 32), tq=_log(rng, 1, 512), tk=_log(rng, 512, 4096),
                    D=rng.choice([64, 128]), nblocks=rng.choice([4, 9, 16]),
                    dtype=rng.choice(["float16", "float32"]), causal=rng.random() < 0.5)
    if kind == "iqa":
        return dict(kind=kind, heads=_log(rng, 2, 32), tq=_log(rng, 1, 64), tk=_log(rng, 512, 4096),
                    D=rng.choice([64, 128]), nblocks=rng.choice([4, 16, 64]),
                    precs=rng.choice(["INT8,INT4_RESIDUAL,FP8", "FP16,INT8", "INT8", "INT4,FP8,SKIP"]))
    if kind == "quantize":
        return dict(kind=kind, pages=_log(rng, 64, 32768), D=rng.choice([64, 128]))
    return dict(kind=kind, B=_log(rng, 1, 32), H=rng.choice([1, 2, 8]), T=_log(rng, 2048, 65536),
                share=rng.choice([0.15, 0.4]))


# --------------------------------------------------------------------------- #
# Inputs, from the seed alone
# --------------------------------------------------------------------------- #

def _gens(seed):
    return (torch.Generator(device="cuda").manual_seed(seed * 7919 + 11), torch.Generator().manual_seed(seed * 6151 + 5))


def _randn(g, shape, dtype=torch.float32):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32).to(dtype)


def _over127(x):
    return x / torch.full((1,), 127.0, dtype=x.dtype, device=x.device)    # a true division


def _page_codes(x, tag):
    """float16 pages -> (codes, scales) in the pools' storage format (absmax / 127 in
    float16, round half to even; INT4: groups of 32 channels)."""
    n, _, D = x.shape
    if tag == INT4:
        y = x.reshape(n, PS, D // 32, 32)
        s = _over127(y.abs().amax(dim=(1, 3), keepdim=True))
        c = (y / s).clamp(-7, 7).round().to(torch.int16).reshape(n, PS, D) + 8
        return (c[..., 0::2] | (c[..., 1::2] << 4)).to(torch.uint8), s.reshape(n, D // 32)
    flat = x.reshape(n, -1)
    s = _over127(flat.abs().amax(dim=1, keepdim=True))
    y = flat / s
    if tag == FP8:
        return y.to(torch.float8_e4m3fn).view(torch.uint8).reshape(x.shape), s.reshape(n)
    if tag == INT8:
        return y.clamp(-127, 127).round().to(torch.int8).reshape(x.shape), s.reshape(n)
    base = y.clamp(-7, 7).round()
    resid = flat.float() - base.float() * s.float()
    s2 = _over127(resid.abs().amax(dim=1, keepdim=True)).clamp(min=1e-8)
    r = (resid / s2).clamp(-7, 7).round()
    packed = ((base.to(torch.int16) + 8) | ((r.to(torch.int16) + 8) << 4)).to(torch.uint8)
    return packed.reshape(x.shape), torch.stack([s.float().reshape(n), s2.reshape(n)], dim=1)


def _page_values(codes, scales, tag):
    """The float64 values of pages stored as _page_codes stores them."""
    n = codes.shape[0]
    if tag == FP16:
        return codes.double()
    if tag == FP8:
        return codes.view(torch.float8_e4m3fn).float().double() * scales.double().view(n, 1, 1)
    if tag == INT8:
        return codes.double() * scales.double().view(n, 1, 1)
    if tag == INT4:
        D = 2 * codes.shape[2]
        v = torch.stack([(codes & 15).to(torch.int16) - 8, (codes >> 4).to(torch.int16) - 8], dim=-1)
        v = v.reshape(n, PS, D // 32, 32).double() * scales.double().view(n, 1, D // 32, 1)
        return v.reshape(n, PS, D)
    s = scales.double()
    return ((codes & 15).double() - 8) * s[:, 0].view(n, 1, 1) + ((codes >> 4).double() - 8) * s[:, 1].view(n, 1, 1)


def _decode_inputs(c, seed):
    g, gc = _gens(seed)
    B, Hq, Hkv, D, W = c["B"], c["Hq"], c["Hkv"], c["D"], c["W"]
    rows = B * Hkv
    per = int(math.ceil(W / c["share"]))
    NP = rows * per
    mix = _MIX[c["mix"]]
    tags = torch.tensor(list(mix), dtype=torch.int32)[torch.multinomial(
        torch.tensor(list(mix.values())), NP, replacement=True, generator=gc)].cuda()
    # each row selects W of its own logical pages, which lie at random in the pool
    table = torch.randperm(NP, generator=gc)[:rows * W].to(torch.int32).reshape(B, Hkv, W).cuda()
    counts = (torch.randint(max(1, W // 2), W + 1, (B, Hkv), generator=gc) if c["ragged"]
              else torch.full((B, Hkv), W)).to(torch.int32).cuda()
    pools = {}
    present = [t for t in (FP16, INT8, FP8, INT4, INT4R) if t in (FP16, INT8) or t in mix]
    for t in present:
        for w in "kv":
            shape = (NP, PS, D // 2 if t == INT4 else D)
            dt = torch.float16 if t == FP16 else (torch.int8 if t == INT8 else torch.uint8)
            pools[w, t] = torch.zeros(shape, dtype=dt, device="cuda")
            if t in (INT8, FP8):
                pools[w, t, "s"] = torch.ones(NP, dtype=torch.float16, device="cuda")
            elif t == INT4:
                pools[w, t, "s"] = torch.ones((NP, D // 32), dtype=torch.float16, device="cuda")
            elif t == INT4R:
                pools[w, t, "s"] = torch.ones((NP, 2), dtype=torch.float32, device="cuda")
    for lo in range(0, NP, 131072):
        hi = min(NP, lo + 131072)
        at = {t: torch.nonzero(tags[lo:hi] == t).flatten() for t in present}
        for w in "kv":
            x = torch.randn((hi - lo, PS, D), generator=g, device="cuda", dtype=torch.float16)
            for t in present:
                if t == FP16:
                    pools[w, t][lo:hi] = x
                elif at[t].numel():
                    codes, scales = _page_codes(x[at[t]], t)
                    pools[w, t][lo + at[t]] = codes
                    pools[w, t, "s"][lo + at[t]] = scales.to(pools[w, t, "s"].dtype)
    q = _randn(g, (B, Hq, D), _DTYPE[c["q"]])
    return q, pools, table, counts, tags


def _latent_inputs(c, seed):
    g, gc = _gens(seed)
    B, W, dqk = c["B"], c["W"], c["dqk"]
    NP = 2 * B * W
    kinds = {"codes": [FP8, INT8], "fp16": [FP16], "mixed": [FP16, FP8, INT8]}[c["pool"]]
    tags = torch.tensor(kinds, dtype=torch.int32)[torch.randint(0, len(kinds), (NP,), generator=gc)].cuda()
    table = torch.randperm(NP, generator=gc)[:B * W].to(torch.int32).reshape(B, W).cuda()
    if c["ragged"]:
        tokens = torch.randint(max(1, PS * W // 2), PS * W + 1, (B,), generator=gc).to(torch.int32)
        counts = (tokens + PS - 1) // PS
        tokens, counts = tokens.cuda(), counts.to(torch.int32).cuda()
    else:
        tokens, counts = None, torch.full((B,), W, dtype=torch.int32, device="cuda")
    x = torch.randn((NP, PS, dqk), generator=g, device="cuda", dtype=torch.float16)
    pools = {}
    for t in kinds:
        if t == FP16:
            pools[t] = x
            continue
        codes, scales = _page_codes(x, t)
        pools[t], pools[t, "s"] = codes, scales
    return _randn(g, (B, c["H"], dqk), _DTYPE[c["q"]]), pools, table, counts, tags, tokens


def _layout(c, seed):
    """Blocks that cover the context, the first one always selected; about a quarter skipped.
    Odd lengths unless the context divides evenly into the blocks."""
    rng = np.random.default_rng(seed * 31 + 7)
    n, T = c["nblocks"], c["tk"]
    if T % n == 0:
        cuts = [T // n * i for i in range(n + 1)]
    else:
        cuts = [0] + sorted(rng.choice(np.arange(1, T), n - 1, replace=False).tolist()) + [T]
    skipped = set(rng.choice(np.arange(1, n), max(1, n // 4), replace=False).tolist())
    blocks = []
    for i in range(n):
        pol = (ia.BlockPolicy.ALWAYS if i == 0 else ia.BlockPolicy.SKIP if i in skipped else ia.BlockPolicy.ATTEND)
        blocks.append(ia.SemanticBlock(f"b{i}", int(cuts[i]), int(cuts[i + 1]), pol,
                                       0.9 if pol == ia.BlockPolicy.ATTEND else None))
    return ia.BlockLayout(blocks)


def _attention_inputs(c, seed):
    g, gc = _gens(seed)
    dt = _DTYPE[c.get("dtype", "float32")]
    lead = (1, c["heads"])
    q = _randn(g, (*lead, c["tq"], c["D"]), dt)
    k = _randn(g, (*lead, c["tk"], c["D"]), dt)
    v = _randn(g, (*lead, c["tk"], c["D"]), dt)
    mask = None
    if c.get("mask"):     # an additive bias with a tenth of the keys shut out, never a row's first key
        mask = _randn(g, (c["tq"], c["tk"]), dt)
        shut = torch.rand((c["tq"], c["tk"]), generator=g, device="cuda") < 0.1
        shut[:, 0] = False
        mask = mask.masked_fill(shut, float("-inf"))
    return q, k, v, mask


class _Assigned:
    """A precision per selected block, by its name."""

    def __init__(self, plan):
        self.plan = plan

    def assign_block_precision(self, block):
        return ia.QuantPolicy(self.plan[block.name])


def _precisions(c, layout):
    names = c["precs"].split(",")
    return {b.name: ia.KVPrecision(names[i % len(names)]) for i, b in enumerate(layout.selected_blocks())}


def _mla_api_inputs(c, seed):
    g, gc = _gens(seed)
    q = _randn(g, (c["B"], c["q_len"], c["dc"]), _DTYPE[c["q"]])
    C = _randn(g, (c["T"], c["dc"]), _DTYPE[c["c"]])
    W = (_randn(g, (c["dc"], c["d_out"])) / math.sqrt(c["dc"])).half()
    ids = torch.randperm(c["T"] // c["page"], generator=gc)[:c["pages"]].to(torch.int32).cuda()
    return q, C, W, ids


_QUANT = (("FP8", FP8), ("INT8", INT8), ("INT4", INT4), ("INT4_RESIDUAL", INT4R))


def _quantize_inputs(c, seed):
    g, gc = _gens(seed)
    n, D = c["pages"], c["D"]
    out = []
    for name, tag in _QUANT:
        x = torch.randn((n, PS, D), generator=g, device="cuda", dtype=torch.float16)
        out.append((name, tag, x, torch.randperm(n, generator=gc).to(torch.int32).cuda()))
    return out


def _routing_inputs(c, seed):
    """Per sequence the routed blocks (16..1024 tokens, a share of the context selected,
    in routed order) and its logical -> physical pages."""
    rng = np.random.default_rng(seed * 17 + 3)
    P = (c["T"] + PS - 1) // PS
    lists = []
    for _ in range(c["B"]):
        cuts, t = [], 0
        while t < c["T"]:
            n = int(rng.integers(16, 1025))
            cuts.append((t, min(c["T"], t + n)))
            t += n
        got, spans = 0, []
        for i in rng.permutation(len(cuts)):
            if got >= c["share"] * c["T"]:
                break
            spans.append((*cuts[i], str(rng.choice(["FP16", "FP8", "INT8", "INT4"], p=[.25, .25, .30, .20]))))
            got += cuts[i][1] - cuts[i][0]
        lists.append(spans)
    NP = c["B"] * P
    table = rng.permutation(NP).astype(np.int32).reshape(c["B"], P)
    return lists, NP, P, table


# --------------------------------------------------------------------------- #
# prepare / run
# --------------------------------------------------------------------------- #

def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind == "decode":
        q, p, table, counts, tags = _decode_inputs(c, seed)
        native = ia.PagePools(int4_group=32)
        for t in (FP8, INT4, INT4R):
            for w in "kv":
                if (w, t) in p:
                    setattr(native, f"{w}_{_NAME[t]}", p[w, t])
                    setattr(native, f"{w}_{_NAME[t]}_scale", p[w, t, "s"])
        args = (p["k", FP16], p["v", FP16], p["k", INT8], p["v", INT8], p["k", INT8, "s"], p["v", INT8, "s"],
                table, counts, tags)
        if c["api"] == "sibling":   # its own tag numbering, -1 past each row's count
            tags = torch.tensor([0, 2, 5, 1, 3, 4], dtype=torch.int32, device="cuda")[tags.long()]
            past = torch.arange(c["W"], device="cuda") >= counts[..., None]
            table = table.masked_fill(past, -1)
            args = args[:6] + (table, counts, tags)
            cfg = IntentQuantKernelConfig(head_dim=c["D"], max_selected_pages=c["W"], block_d=c["D"])
        else:
            q = q[:, :, None, :]
            args = args[:6] + (table, tags, counts)
            cfg = ia.FusedDecodeConfig(head_dim=c["D"], max_selected_pages=c["W"], block_d=c["D"])
        return dict(kind=kind, api=c["api"], q=q, args=args, cfg=cfg, native=native)
    if kind == "mla_paged":
        q, p, table, counts, tags, tokens = _latent_inputs(c, seed)
        pools = ia.LatentPools(c_fp16=p.get(FP16), c_fp8=p.get(FP8), c_int8=p.get(INT8),
                               c_fp8_scale=p.get((FP8, "s")), c_int8_scale=p.get((INT8, "s")))
        return dict(kind=kind, q=q, pools=pools, table=table, counts=counts, tags=tags, tokens=tokens, dv=c["dv"])
    if kind == "mla_api":
        q, C, W, ids = _mla_api_inputs(c, seed)
        return dict(kind=kind, q=q, C=C, W=W, ids=ids, page=c["page"])
    if kind == "dense":
        q, k, v, mask = _attention_inputs(c, seed)
        return dict(kind=kind, q=q, k=k, v=v, mask=mask, causal=c["causal"])
    if kind == "blocks":
        q, k, v, _ = _attention_inputs(c, seed)
        return dict(kind=kind, q=q, k=k, v=v, layout=_layout(c, seed), causal=c["causal"])
    if kind == "iqa":
        q, k, v, _ = _attention_inputs(c, seed)
        layout = _layout(c, seed)
        return dict(kind=kind, q=q, k=k, v=v, layout=layout, quantizer=_Assigned(_precisions(c, layout)))
    if kind == "quantize":
        jobs = []
        for name, tag, x, dst in _quantize_inputs(c, seed):
            n, D = c["pages"], c["D"]
            codes = torch.zeros((n, PS, D // 2 if tag == INT4 else D), device="cuda",
                                dtype=torch.int8 if tag == INT8 else torch.uint8)
            scales = (torch.zeros((n, D // 32), dtype=torch.float16, device="cuda") if tag == INT4 else
                      torch.zeros((n, 2), device="cuda") if tag == INT4R else
                      torch.zeros(n, dtype=torch.float16, device="cuda"))
            jobs.append((name, x, dst, codes, scales))
        return dict(kind=kind, jobs=jobs)
    lists, NP, P, table = _routing_inputs(c, seed)
    routed = [[ia.RoutedBlock(f"b{i}", s, e, ia.BlockPolicy.ATTEND, 0.5, ia.BlockDecision.SELECT,
                              ia.KVPrecision(p), "scored") for i, (s, e, p) in enumerate(spans)] for spans in lists]
    return dict(kind=kind, routed=routed, NP=NP, B=c["B"], H=c["H"], table=torch.from_numpy(table).cuda(),
                cfg=ia.FusedDecodeConfig(max_selected_pages=_table_width(c)))


def _table_width(c):
    # the selected share, the last block's overshoot and a page shared at either end of each block
    return int(c["share"] * c["T"]) // PS + 64 + 2 * (c["T"] // 400)


def run(state):
    s, kind = state, state["kind"]
    if kind == "decode":
        if s["api"] == "sibling":
            return intent_quant_decode_attention_triton(s["q"], *s["args"], config=s["cfg"], native_pools=s["native"])
        return ia.fused_selected_quant_decode(s["q"], *s["args"], s["cfg"], native_pools=s["native"])
    if kind == "mla_paged":
        return ia.mla_paged_decode(s["q"], s["pools"], s["table"], s["counts"], s["tags"], v_dim=s["dv"],
                                   valid_tokens=s["tokens"])
    if kind == "mla_api":
        return ia.mla_decode_triton(s["q"], s["C"], s["W"], s["ids"], s["page"])
    if kind == "dense":
        return ia.dense_attention(s["q"], s["k"], s["v"], causal=s["causal"], mask=s["mask"])
    if kind == "blocks":
        return ia.semantic_block_attention(s["q"], s["k"], s["v"], s["layout"], causal=s["causal"])
    if kind == "iqa":
        return ia.intent_quant_attention_reference(s["q"], s["k"], s["v"], s["layout"], s["quantizer"])
    if kind == "quantize":
        return [ia.quantize_pages(x, name, codes=codes, scales=scales, dst_pages=dst)
                for name, x, dst, codes, scales in s["jobs"]]
    return ia.routing_to_kernel_tensors(s["routed"], PS, s["NP"], s["B"], s["H"], s["cfg"], native_precisions=True,
                                        block_table=s["table"])


# --------------------------------------------------------------------------- #
# work / tolerance / exact
# --------------------------------------------------------------------------- #

def _selected_tokens(c):
    """Selected tokens of _layout, as an expectation over the seeds where the cuts are random."""
    n = c["nblocks"]
    return int(c["tk"] * (n - max(1, n // 4)) / n)


def work(case):
    c, kind = case, case["kind"]
    if kind == "decode":
        fill = 0.75 if c["ragged"] else 1.0
        pages = c["B"] * c["Hkv"] * c["W"] * fill
        D = c["D"]
        per = {FP16: 4 * PS * D, FP8: 2 * PS * D + 4, INT8: 2 * PS * D + 4, INT4: PS * D + 4 * (D // 32),
               INT4R: 2 * PS * D + 16, SKIP: 0}
        mix = _MIX[c["mix"]]
        out = _SIZE[c["q"]] if c["api"] == "sibling" else 2
        live = sum(f for t, f in mix.items() if t != SKIP)
        return {"bytes": pages * (8 + sum(f * per[t] for t, f in mix.items()))
                + c["B"] * c["Hq"] * D * (_SIZE[c["q"]] + out) + 4 * c["B"] * c["Hkv"],
                "flops": 4 * pages * live * PS * D * (c["Hq"] // c["Hkv"])}
    if kind == "mla_paged":
        pages = c["B"] * c["W"] * (0.75 if c["ragged"] else 1.0)
        per = {"codes": 1.0, "fp16": 2.0, "mixed": 4 / 3}[c["pool"]] * PS * c["dqk"]
        return {"bytes": pages * (per + 10) + c["B"] * c["H"] * (c["dqk"] + c["dv"]) * _SIZE[c["q"]],
                "flops": 2 * pages * PS * c["H"] * (c["dqk"] + c["dv"])}
    if kind == "mla_api":
        rows, keys = c["B"] * c["q_len"], c["pages"] * c["page"]
        return {"bytes": keys * c["dc"] * _SIZE[c["c"]] + 2 * c["dc"] * c["d_out"]
                + rows * (c["dc"] + c["d_out"]) * _SIZE[c["q"]] + 4 * c["pages"],
                "flops": 4 * rows * keys * c["dc"] + 2 * rows * c["dc"] * c["d_out"]}
    if kind in ("dense", "blocks", "iqa"):
        keys = c["tk"] if kind == "dense" else _selected_tokens(c)
        size = _SIZE[c.get("dtype", "float32")]
        pairs = c["tq"] * keys
        if c.get("causal"):     # query i sees the keys at positions 0 .. i
            n = min(c["tq"], c["tk"])
            pairs = (n * (n + 1) // 2 + (c["tq"] - n) * n) * keys // c["tk"]
            keys = keys * n // c["tk"]
        return {"bytes": c["heads"] * c["D"] * size * 2 * (c["tq"] + keys) + (c["tq"] * c["tk"] * size if c.get("mask") else 0),
                "flops": 4 * c["heads"] * pairs * c["D"]}
    if kind == "quantize":
        n, D = c["pages"], c["D"]
        page = 2 * PS * D + 4
        return {"bytes": n * (4 * page + 3 * PS * D + PS * D // 2 + 2 + 2 + 2 * (D // 32) + 8), "flops": 0}
    pages = c["B"] * c["share"] * c["T"] / PS
    NP = c["B"] * ((c["T"] + PS - 1) // PS)
    return {"bytes": 4 * (pages + c["B"] * c["H"] * (_table_width(c) + 1) + NP), "flops": 0}


def tolerance(case):
    kind = case["kind"]
    if kind in ("quantize", "tables"):
        return "exact"
    # four times the error against exact() that a one-rounding-per-output path shows:
    # 2e-4 for float16 outputs, 1.7e-3 for bfloat16, 6e-7 for float32 sums throughout
    out = case.get("q", case.get("dtype", "float32"))
    if kind == "decode" and case["api"] == "fused":
        out = "float16"
    if out == "float32" and kind in ("decode", "mla_paged"):
        return {"rel": 1e-3}     # float16 matrix operands (weights, quantised values) under a float32 output
    return {"rel": {"float16": 1.2e-3, "bfloat16": 7e-3, "float32": 3e-6}[out]}


def _softmax_attention(q, k, v, bias=None):
    """softmax(q k^T / sqrt(D) + bias) v in float64, a head at a time."""
    out = torch.empty((*q.shape[:-1], v.shape[-1]), dtype=torch.float64, device=q.device)
    for h in range(q.shape[1]):
        s = q[0, h].double() @ k[0, h].double().T / math.sqrt(q.shape[-1])
        if bias is not None:
            s = s + bias
        out[0, h] = torch.softmax(s, dim=-1) @ v[0, h].double()
    return out


def _fake_quant(x, prec):
    """One block's fake-quant reconstruction, one scale per channel, in the
    float32 arithmetic that defines it."""
    P = ia.KVPrecision
    if prec == P.FP16:
        return x.half().float()
    if prec == P.SKIP:
        return torch.zeros_like(x)

    def scale(t):
        return _over127(t.abs().amax(dim=tuple(range(t.dim() - 1)), keepdim=True)).clamp(min=1e-8)
    s = scale(x)
    if prec == P.FP8:
        return (x / s).to(torch.float8_e4m3fn).float() * s
    if prec == P.INT8:
        return (x / s).clamp(-127, 127).round() * s
    base = (x / s).clamp(-7, 7).round() * s
    if prec == P.INT4:
        return base
    s2 = scale(x - base)
    return base + ((x - base) / s2).clamp(-7, 7).round() * s2


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "decode":
        q, p, table, counts, tags = _decode_inputs(c, seed)
        B, Hq, Hkv, D = c["B"], c["Hq"], c["Hkv"], c["D"]
        G = Hq // Hkv
        out = torch.zeros((B, Hq, D), dtype=torch.float64, device="cuda")
        counts = counts.tolist()
        for b in range(B):
            for h in range(Hkv):
                ids = table[b, h, :counts[b][h]].long()
                tg = tags[ids]
                ids, tg = ids[tg != SKIP], tg[tg != SKIP]
                if ids.numel() == 0:
                    continue
                kv = []
                for w in "kv":
                    x = torch.empty((ids.numel(), PS, D), dtype=torch.float64, device="cuda")
                    for t in _MIX[c["mix"]]:
                        at = torch.nonzero(tg == t).flatten()
                        if t != SKIP and at.numel():
                            sc = None if t == FP16 else p[w, t, "s"][ids[at]]
                            x[at] = _page_values(p[w, t][ids[at]], sc, t)
                    kv.append(x.reshape(-1, D))
                s = q[b, h * G:(h + 1) * G].double() @ kv[0].T / math.sqrt(D)
                out[b, h * G:(h + 1) * G] = torch.softmax(s, dim=-1) @ kv[1]
        return out if c["api"] == "sibling" else out[:, :, None, :]
    if kind == "mla_paged":
        q, p, table, counts, tags, tokens = _latent_inputs(c, seed)
        out = torch.zeros((c["B"], c["H"], c["dv"]), dtype=torch.float64, device="cuda")
        counts = counts.tolist()
        for b in range(c["B"]):
            ids = table[b, :counts[b]].long()
            x = torch.empty((ids.numel(), PS, c["dqk"]), dtype=torch.float64, device="cuda")
            for t in (FP16, FP8, INT8):
                at = torch.nonzero(tags[ids] == t).flatten()
                if at.numel():
                    x[at] = _page_values(p[t][ids[at]], None if t == FP16 else p[t, "s"][ids[at]], t)
            x = x.reshape(-1, c["dqk"])
            if tokens is not None:
                x = x[:int(tokens[b])]
            s = q[b].double() @ x.T / math.sqrt(c["dqk"])
            out[b] = torch.softmax(s, dim=-1) @ x[:, :c["dv"]]
        return out
    if kind == "mla_api":
        q, C, W, ids = _mla_api_inputs(c, seed)
        rows = (ids.long()[:, None] * c["page"] + torch.arange(c["page"], device="cuda")).flatten()
        x = C[rows].double()
        s = q.double() @ x.T / math.sqrt(c["dc"])
        return torch.softmax(s, dim=-1) @ x @ W.double()
    if kind == "dense":
        q, k, v, mask = _attention_inputs(c, seed)
        bias = torch.zeros((c["tq"], c["tk"]), dtype=torch.float64, device="cuda")
        if c["causal"]:
            bias += torch.triu(torch.full_like(bias, float("-inf")), diagonal=1)
        if mask is not None:
            bias += mask.double()
        return _softmax_attention(q, k, v, bias)
    if kind == "blocks":
        q, k, v, _ = _attention_inputs(c, seed)
        at = torch.cat([torch.arange(b.start, b.end) for b in _layout(c, seed).selected_blocks()]).cuda()
        bias = None
        if c["causal"]:
            hidden = torch.arange(c["tq"], device="cuda")[:, None] < at[None, :]
            bias = torch.zeros(hidden.shape, dtype=torch.float64, device="cuda").masked_fill(hidden, float("-inf"))
        return _softmax_attention(q, k[:, :, at], v[:, :, at], bias)
    if kind == "iqa":
        q, k, v, _ = _attention_inputs(c, seed)
        layout = _layout(c, seed)
        plan = _precisions(c, layout)
        rec = [torch.cat([_fake_quant(x[:, :, b.start:b.end], plan[b.name]) for b in layout.selected_blocks()], dim=2)
               for x in (k, v)]
        return _softmax_attention(q, *rec)
    if kind == "quantize":
        out = []
        for name, tag, x, dst in _quantize_inputs(c, seed):
            codes, scales = _page_codes(x, tag)
            at = torch.argsort(dst.long())
            out.append((codes[at], scales[at].float() if tag == INT4R else scales[at]))
        return out
    lists, NP, P, table = _routing_inputs(c, seed)
    W = _table_width(c)
    pages = np.zeros((c["B"], c["H"], W), dtype=np.int32)
    counts = np.zeros((c["B"], c["H"]), dtype=np.int32)
    prec = np.full(NP, FP16, dtype=np.int32)
    tag = {"FP16": FP16, "FP8": FP8, "INT8": INT8, "INT4": INT4}
    for b, spans in enumerate(lists):
        seen = {}
        for s, e, p in spans:
            for pg in range(s // PS, (e - 1) // PS + 1):
                seen.setdefault(pg, tag[p])
        ids = [int(table[b, pg]) for pg in seen]
        for i, t in zip(ids, seen.values()):
            prec[i] = t
        pages[b, :, :min(W, len(ids))] = ids[:W]
        counts[b] = min(W, len(ids))
    return tuple(torch.from_numpy(x) for x in (pages, prec, counts))
