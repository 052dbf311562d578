"""dense_attention on the matrix-core form (csrc/dense_matrix.h): the edges of its
query and key tiles, padded widths, every mask form, strided and broadcast operands,
and non-finite values, against the float64 oracle and against the row form (the
library without a workspace), which the form has to agree with value for value up
to rounding and NaN / infinity for NaN / infinity."""
import numpy as np
import pytest
import torch

from oracle import attention as A

pytestmark = pytest.mark.gpu

DT = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
# float32: 2e-5 as elsewhere for float32 sums; 16-bit outputs: half an ulp of values
# of at most 4 besides (2^-10 and 2^-7 relative spacing halves)
TOL = {"f16": 2e-5 + 4 * 2 ** -11, "bf16": 2e-5 + 4 * 2 ** -8, "f32": 2e-5}


def _rows_form(monkeypatch, *a, **kw):
    from intent_attention import _native as N
    from intent_attention import dense_attention
    with monkeypatch.context() as mp:
        mp.setattr(N, "dense_attention_workspace", lambda args: 0)
        return dense_attention(*a, **kw)


def _qkv(seed, lead, tq, tk, d, dv, dt):
    g = torch.Generator().manual_seed(seed)
    mk = lambda *s: torch.randn(*s, generator=g).to(DT[dt])  # noqa: E731
    return mk(*lead, tq, d), mk(*lead, tk, d), mk(*lead, tk, dv), g


def _check(got, want, dt, what):
    o = got.double().cpu().numpy()
    err = np.abs(o - want).max()
    print(f"[gpu-case] {what}: max abs err {err:.2e}", flush=True)
    assert err <= TOL[dt], what


# (tq, tk, d, dv): one below, at and one above the query tiles (32, 64, 128 rows) and the
# key tiles (64 or 128 keys), the smallest widths, padded ones, unequal ones, the widest
SHAPES = [(31, 64, 64, 64), (32, 65, 64, 64), (33, 63, 128, 128), (64, 129, 128, 64), (65, 127, 64, 128),
          (127, 300, 128, 128), (128, 1, 64, 64), (129, 513, 96, 96), (257, 257, 72, 80), (40, 200, 8, 16),
          (100, 130, 192, 136), (70, 190, 256, 200), (2, 1500, 128, 128), (5, 700, 64, 64)]


@pytest.mark.parametrize("dt", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("tq,tk,d,dv", SHAPES)
def test_tile_edges(tq, tk, d, dv, dt):
    from intent_attention import dense_attention
    lead = (2, max(2, -(-50000 // (2 * tq * tk))))
    q, k, v, _ = _qkv(tq * 1000 + tk, lead, tq, tk, d, dv, dt)
    n = lambda *x: [t.double().numpy() for t in x]  # noqa: E731
    c = lambda *x: [t.cuda() for t in x]  # noqa: E731
    for causal in (False, True):
        _check(dense_attention(*c(q, k, v), causal=causal), A.dense_attention_masked(*n(q, k, v), causal=causal), dt,
               f"{dt} {lead} {tq}x{tk}x{d}/{dv} causal={causal}")


@pytest.mark.parametrize("dt", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("tq,tk", [(12, 900), (130, 200)])
def test_masks_positions_and_layouts(tq, tk, dt, monkeypatch):
    from intent_attention import dense_attention
    q, k, v, g = _qkv(7, (2, 4), tq, tk, 64, 64, dt)
    mask = torch.randn(tq, tk, generator=g)
    mask[torch.rand(tq, tk, generator=g) < 0.3] = float("-inf")
    mask[:, 3] = 0.0
    low = torch.zeros(tq, tk).to(DT[dt])
    low[:, tk // 2:] = torch.finfo(DT[dt]).min
    low[1] = torch.finfo(DT[dt]).min            # a whole row of the lowest value: still a softmax
    dead = torch.zeros(tq, tk).to(DT[dt])
    dead[2] = float("-inf")                     # a row with nothing to attend: NaN
    pos = torch.sort(torch.randperm(3 * tk, generator=g)[:tk]).values
    pos[0] = 0
    bools = torch.rand(2, 1, tq, tk, generator=g) < 0.5
    cases = [dict(mask=mask.to(DT[dt])), dict(mask=low), dict(mask=dead), dict(mask=bools),
             dict(causal=True, mask=mask.to(DT[dt])), dict(causal=True, original_kv_positions=pos),
             dict(causal=True, original_kv_positions=pos.flip(0))]
    qc, kc, vc = q.cuda(), k.cuda(), v.cuda()
    # [B, T, H, D] storage, and K / V broadcast over the heads
    swapped = [x.transpose(1, 2).contiguous().transpose(1, 2) for x in (qc, kc, vc)]
    shared = [qc, kc[:, :1], vc[:, :1]]
    for kw in cases:
        kw = {n: (x.cuda() if isinstance(x, torch.Tensor) else x) for n, x in kw.items()}
        for ops in ((qc, kc, vc), swapped, shared):
            got, want = dense_attention(*ops, **kw), _rows_form(monkeypatch, *ops, **kw)
            assert torch.equal(torch.isnan(got), torch.isnan(want)), sorted(kw)
            live = ~torch.isnan(want)
            assert float((got[live].double() - want[live].double()).abs().max()) <= 2 * TOL[dt], sorted(kw)


@pytest.mark.parametrize("dt", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("tq,tk,d", [(128, 300, 64), (300, 300, 128), (16, 2200, 64), (1100, 700, 64)])
def test_nonfinite_values_as_the_row_form(tq, tk, d, dt, monkeypatch):
    """Infinities, NaN and values whose scores overflow, in visible and in causally hidden
    keys, give what the plain sums give: the tiles past the diagonal and the split of
    the weights must not hide or invent one."""
    from intent_attention import dense_attention
    big = 60000.0 if dt == "f16" else 1e37
    for where, value in (("k", np.inf), ("k", np.nan), ("v", np.inf), ("v", -np.inf), ("v", np.nan), ("k", big),
                         ("q", np.inf), ("q", big)):
        for causal in (False, True):
            q, k, v, _ = _qkv(11, (1, 2), tq, tk, d, d, dt)
            x, at = {"q": (q, tq // 2), "k": (k, tk - 5), "v": (v, tk - 5)}[where]
            x[0, 0, at, 3 if abs(value) != big else slice(None)] = value
            ops = [t.cuda() for t in (q, k, v)]
            got, want = dense_attention(*ops, causal=causal), _rows_form(monkeypatch, *ops, causal=causal)
            what = f"{where}={value} causal={causal}"
            assert torch.equal(torch.isnan(got), torch.isnan(want)), what
            assert torch.equal(torch.isinf(got), torch.isinf(want)), what
            live = torch.isfinite(want)
            assert float((got[live].double() - want[live].double()).abs().max()) <= 2 * TOL[dt], what


def test_replays_from_a_graph():
    from intent_attention import dense_attention
    q, k, v, g = _qkv(3, (1, 8), 200, 333, 128, 128, "f16")
    qc, kc, vc = q.cuda(), k.cuda(), v.cuda()
    eager = dense_attention(qc, kc, vc, causal=True)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = dense_attention(qc, kc, vc, causal=True)
    for i in range(3):
        qc.copy_(torch.randn(q.shape, generator=g).half())
        graph.replay()
        want = dense_attention(qc, kc, vc, causal=True)
        torch.cuda.synchronize()
        assert torch.equal(out, want) and not torch.equal(out, eager), i


@pytest.mark.parametrize("dt", ["f16", "bf16", "f32"])
def test_short_calls_replay_from_a_graph(dt):
    """A short call has no workspace of its own, and its second walk runs when a replay's inputs ask
    for it: finite inputs, an infinity, finite ones again."""
    from intent_attention import dense_attention
    q, k, v, g = _qkv(5, (4, 40), 20, 200, 64, 64, dt)
    qc, kc, vc = q.cuda(), k.cuda(), v.cuda()
    dense_attention(qc, kc, vc)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = dense_attention(qc, kc, vc)
    for i in range(4):
        qc.copy_(torch.randn(q.shape, generator=g).to(DT[dt]))
        vc[1, 3, 199, 7] = float("inf") if i % 2 else 1.0
        graph.replay()
        want = dense_attention(qc, kc, vc)
        torch.cuda.synchronize()
        assert torch.equal(out, want), i
        assert bool(torch.isposinf(out[1, 3, :, 7]).all()) == bool(i % 2) and int(torch.isinf(out).sum()) == 20 * (i % 2)


# rows form (1 row, few pairs), split rows, and the three wave shapes of the matrix form; head
# dims with and without 16-byte rows
@pytest.mark.parametrize("dt", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("tq,d", [(1, 64), (3, 20), (5, 128), (40, 64), (128, 64), (130, 96)])
def test_selected_blocks_read_in_place(tq, d, dt):
    """Keys read through the selected tokens' index are bit for bit the gathered keys' result,
    NaN and infinity in and outside the selection included."""
    from intent_attention import BlockLayout, BlockPolicy, SemanticBlock, dense_attention, semantic_block_attention
    spans = [(0, 3), (5, 64), (64, 65), (130, 700), (901, 1000)]
    layout = BlockLayout([SemanticBlock(f"b{i}", s, e, BlockPolicy.ALWAYS) for i, (s, e) in enumerate(spans)])
    sel = torch.tensor([t for s, e in spans for t in range(s, e)]).cuda()
    lead = (2, 8)
    q, k, v, _ = (x.cuda() if isinstance(x, torch.Tensor) else x for x in _qkv(tq + d, lead, tq, 1000, d, d, dt))
    k[:, :, 800] = float("nan")             # not selected
    v[:, :, 4] = float("inf")
    for case in ("finite", "inf in v", "strided"):
        if case == "inf in v":
            v[1, 3, 699] = float("inf")
        if case == "strided":               # not read in place
            k = k.transpose(0, 1).contiguous().transpose(0, 1)
        for causal in (False, True):
            want = dense_attention(q, k.index_select(-2, sel), v.index_select(-2, sel), causal=causal,
                                   original_kv_positions=sel)
            got, debug = semantic_block_attention(q, k, v, layout, causal=causal, return_debug=True)
            assert torch.equal(torch.nan_to_num(got, 7.0, 8.0, -8.0), torch.nan_to_num(want, 7.0, 8.0, -8.0)), case
            assert debug["selected_kv_tokens"] == debug["selected_token_count"] == sel.numel()
            if case == "finite" and not causal:
                assert bool(got.isfinite().all())


# both sides of the eight-wave rule (256 workgroups; causal 512; more than 128 keys), with
# ragged rows and keys; 8 query tiles x 65 heads is one group per XCD and a remainder
@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("heads,t,tk,d", [(64, 512, 512, 64), (129, 130, 257, 96), (128, 129, 129, 128),
                                          (257, 66, 300, 64), (65, 1000, 1000, 64), (3, 700, 128, 128)])
def test_waves_per_workgroup(heads, t, tk, d, dt, monkeypatch):
    from intent_attention import dense_attention
    q, k, v, _ = _qkv(heads + t, (heads,), t, tk, d, d, dt)
    q, k, v = q.cuda(), k.cuda(), v.cuda()
    for causal in (False, True):
        got = dense_attention(q, k, v, causal=causal)
        rows = _rows_form(monkeypatch, q, k, v, causal=causal)
        _check(got, rows.double().cpu().numpy(), dt, f"{dt} {heads}x{t}x{tk}x{d} causal={causal}")
        # one head in float64
        n = lambda x: x[heads // 2:heads // 2 + 1].double().cpu().numpy()  # noqa: E731
        _check(got[heads // 2:heads // 2 + 1], A.dense_attention_masked(n(q), n(k), n(v), causal=causal), dt, "one head")


# key counts one short of a 32- or 128-key tile, one past it, and whole tiles; the wave shapes of
# few, some and many query rows, keys split over workgroups (2 to 8 heads) and not, short calls
# (up to 256 keys of a wave x 64 dims) and long ones
@pytest.mark.parametrize("dt", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("heads,tq,tk,d", [(8, 8, 1055, 64), (2, 40, 1025, 64), (2, 128, 1057, 64), (300, 8, 159, 64),
                                           (300, 8, 161, 64), (300, 33, 65, 64), (300, 130, 33, 64), (2, 128, 257, 64),
                                           (64, 20, 129, 128), (40, 60, 95, 96), (130, 150, 128, 128),
                                           (260, 130, 400, 128)])
def test_special_values_in_the_last_key(heads, tq, tk, d, dt, monkeypatch):
    """The last key's row stands in for the keys that fill up its tile: whatever it holds, the
    result is the row form's. Its score is up to 2^7 above the others', as far as the
    running maximum may lag, so a large finite value must not overflow on the way either."""
    from intent_attention import BlockLayout, BlockPolicy, SemanticBlock, dense_attention, semantic_block_attention
    q, k, v, g = _qkv(heads + tk, (heads,), tq, tk, d, d, dt)
    q[..., 0], k[:, :-1] = 4.0, k[:, :-1] * 0.1
    k[:, -1] = 0.0
    k[:, -1, 0] = 9.0 / 8 * d ** 0.5                   # 4 * 9 / 8 log2(e) = 6.5
    big = 60000.0 if dt == "f16" else 1e37
    mask = torch.zeros(tq, tk).to(DT[dt])
    mask[:, 5] = float("-inf")
    pos = torch.arange(tk)
    layout = BlockLayout([SemanticBlock("a", 0, tk, BlockPolicy.ALWAYS)])
    forms = [dict(), dict(mask=mask.cuda()), dict(causal=True, original_kv_positions=pos.flip(0).cuda()), dict(causal=True)]
    q, k, v = q.cuda(), k.cuda(), v.cuda()
    for value in (np.inf, -np.inf, np.nan, big, -big):
        v[0, -1, 3], v[1, -1, :] = value, abs(value)
        for i, kw in enumerate(forms + [None]):
            want = _rows_form(monkeypatch, q, k, v, **(kw or {}))
            got = semantic_block_attention(q, k, v, layout) if kw is None else dense_attention(q, k, v, **kw)
            what = f"{value} form {i}"
            for f in (torch.isnan, torch.isposinf, torch.isneginf):
                assert torch.equal(f(got), f(want)), what
            live = torch.isfinite(want)
            scale = want[live].double().abs().clamp(min=1)
            assert float(((got[live].double() - want[live].double()) / scale).abs().max()) <= 2 * TOL[dt], what


@pytest.mark.parametrize("mask", [False, True])
@pytest.mark.parametrize("tq,tk", [(32, 700), (64, 300), (200, 130)])
def test_small_float16_weights(tq, tk, mask):
    """Keys whose weights are 2^-14 to 2^-30 of the largest, with values that make up for it: the
    weights keep what they had in float32 down to 2^-37 of the largest one (half the smallest
    float16 step after the 2^12 they are kept at), the output its own rounding of 2^-11."""
    from intent_attention import dense_attention
    g = torch.Generator().manual_seed(tq)
    q = torch.zeros(1, 2, tq, 64)
    q[..., 0] = torch.linspace(10, 21, tq).half().float()
    k, v = torch.randn(1, 2, tk, 64, generator=g) * 0.3, 30000 + 30000 * torch.rand(1, 2, tk, 64, generator=g)
    k[..., 0], k[:, :, 40, 0] = torch.rand(1, 2, tk, generator=g) * 0.2, 8.0
    v[:, :, 40] = 0.0
    q, k, v = q.half(), k.half(), v.half()
    m = torch.zeros(tq, tk).half() if mask else None
    got = dense_attention(q.cuda(), k.cuda(), v.cuda(), mask=None if m is None else m.cuda()).double().cpu()
    p = torch.softmax(q.double() @ k.double().transpose(-1, -2) / 8, -1)
    want = p @ v.double()
    # float32 sums besides (2e-5 as above), of the scores too: 21 * 2^-22
    bound = want.abs() * (2 ** -11 + 4e-5) + 2 ** -37 * p.amax(-1, keepdim=True) * v.double().abs().sum(-2, keepdim=True)
    worst = float(((got - want).abs() / bound).max())
    print(f"[gpu-case] {tq}x{tk} mask={mask}: error / bound {worst:.2f}", flush=True)
    assert worst <= 1.0
