"""mla_decode_triton's latent context on the matrix-core form (csrc/mla_rows_matrix.h):
the edges of its 32-row, 32-key and 32-dim tiles, a ragged last page, padded widths,
query and latent dtypes and strides, against float64 and against the rows form (one
query row at a time takes it), NaN and infinities included."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _ref(q, C, ids, ps):
    rows = torch.cat([torch.arange(p * ps, min((p + 1) * ps, C.shape[0])) for p in ids.tolist()]).to(C.device)
    x = C[rows].double()
    s = q.double() @ x.T / q.shape[-1] ** 0.5
    return torch.softmax(s, -1) @ x


# (batch, q_len, d_c, page size, pages listed, rows of C): one tile and its neighbours,
# a last page cut short, widths that pad a wave's part or leave waves idle, the widest
CASES = [(4, 1, 64, 16, 40, 1000), (31, 1, 128, 32, 33, 2000), (32, 1, 128, 31, 34, 1100), (33, 1, 136, 64, 30, 3000),
         (5, 7, 256, 16, 70, 1111), (32, 2, 512, 64, 33, 4096), (64, 1, 576, 64, 33, 2100), (40, 4, 576, 7, 130, 909),
         (97, 1, 640, 64, 40, 2560), (70, 2, 768, 48, 50, 2400)]


@pytest.mark.parametrize("q_dt,c_dt", [("float32", "float16"), ("float16", "bfloat16"), ("bfloat16", "float32")])
@pytest.mark.parametrize("B,T,dc,ps,n,rows", CASES)
def test_against_float64(B, T, dc, ps, n, rows, q_dt, c_dt):
    from intent_attention.triton_mla_decode import mla_latent_context
    g = torch.Generator().manual_seed(B * 100 + dc)
    q = torch.randn(B, T, dc, generator=g).to(getattr(torch, q_dt)).cuda()
    C = torch.randn(rows, dc, generator=g).to(getattr(torch, c_dt)).cuda()
    pages = -(-rows // ps)
    ids = torch.cat([torch.tensor([pages - 1]), torch.randint(0, pages, (n - 1,), generator=g)]).to(torch.int32).cuda()
    wide = torch.randn(rows, dc + 8, generator=g).to(C.dtype).cuda()
    wide[:, :dc] = C
    for qq, cc in ((q, C), (q.transpose(0, 1).contiguous().transpose(0, 1), wide[:, :dc])):
        got = mla_latent_context(qq, cc, ids, ps)
        ref = _ref(q, C, ids, ps)
        err = float((got.double() - ref).abs().max() / ref.abs().max())
        print(f"[gpu-case] {B}x{T}x{dc} pages of {ps}, {q_dt}/{c_dt}: {err:.2e}", flush=True)
        assert err <= 2e-5          # float32 sums, as the rows form's tests


@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan"), 1e37])
def test_nonfinite_latents_as_the_rows_form(value):
    from intent_attention.triton_mla_decode import mla_latent_context
    g = torch.Generator().manual_seed(1)
    q, C = torch.randn(40, 1, 128, generator=g).cuda(), torch.randn(1000, 128, generator=g).cuda()
    C[333, 5] = value
    ids = torch.arange(10, dtype=torch.int32).cuda()
    got = mla_latent_context(q, C, ids, 64)
    want = torch.cat([mla_latent_context(q[i:i + 1], C, ids, 64) for i in range(q.shape[0])])
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got), torch.isinf(want))
    live = torch.isfinite(want)
    assert float((got[live] - want[live]).abs().max()) <= 2e-5 * max(1.0, float(want[live].abs().max()))


@pytest.mark.parametrize("dc", [128, 512, 768])
@pytest.mark.parametrize("c_dt", ["float32", "bfloat16"])
def test_large_latents_that_stay_finite(dc, c_dt):
    """A latent of 1e37 that the scores do not see (its query dim is zero), in a key that scores 2^6
    above the tile before it: its weight must not pass 1 on the way to a context that is finite."""
    from intent_attention.triton_mla_decode import mla_latent_context
    g = torch.Generator().manual_seed(dc)
    n = 9216 if dc == 768 else 1152            # with and without the keys split over workgroups
    B = 40 if dc == 768 else 9000
    q, C = torch.randn(B, 1, dc, generator=g), torch.randn(n, dc, generator=g) * 0.1
    q[..., 0], q[..., 5] = 8.0, 0.0
    C[35] = 0.0
    C[35, 0], C[35, 5] = 4.3 * dc ** 0.5 / 8, 1e37       # exp(4.3) = 2^6.2
    q, C = q.cuda(), C.to(getattr(torch, c_dt)).cuda()
    ids = torch.arange(n // 64, dtype=torch.int32).cuda()
    got = mla_latent_context(q, C, ids, 64)
    want = _ref(q, C, ids, 64)
    assert bool(got.isfinite().all())
    assert float(((got.double() - want).abs() / want.abs().clamp(min=1)).max()) <= 2e-5


def test_without_a_workspace_few_rows_take_the_rows_form():
    """A C caller may pass no workspace; the keys are not split then, and 32 rows go to the
    rows form, as 15 do: each row bit for bit the same in both calls."""
    from intent_attention import _native as N
    from intent_attention.decode_core import current_stream_handle
    g = torch.Generator().manual_seed(2)
    q, C = torch.randn(32, 1, 576, generator=g).cuda(), torch.randn(8192, 576, generator=g).half().cuda()
    ids = torch.arange(128, dtype=torch.int32).cuda()
    out = []
    for rows in (15, 32):
        ctx = torch.empty(rows, 1, 576, device="cuda")
        a = N.MlaRowsArgs()
        a.batch, a.q_len, a.latent_dim, a.page_size, a.num_selected, a.num_rows = rows, 1, 576, 64, 128, 8192
        a.q, a.q_dtype, a.q_stride_b, a.q_stride_t = q.data_ptr(), N.DTYPE_F32, 576, 576
        a.latents, a.latent_dtype, a.latent_stride = C.data_ptr(), N.DTYPE_F16, 576
        a.page_ids, a.context, a.sm_scale = ids.data_ptr(), ctx.data_ptr(), 1 / 24.0
        N.mla_decode_rows(a, current_stream_handle(ctx.device))
        out.append(ctx)
    assert torch.equal(out[0], out[1][:15])
    ref = _ref(q, C, ids, 64)
    assert float((out[1].double() - ref).abs().max() / ref.abs().max()) <= 2e-5
