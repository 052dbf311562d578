"""mla_decode_triton's projection kernel (csrc/mla_project.h): row counts around its 32-row
tiles and the most it takes, latent widths from one group of eight to the widest, W's
dtypes and row strides, the output dtypes, and the forms of W that stay with torch."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _case(rows, dc, d_out, w_dt, q_dt, seed=0):
    g = torch.Generator().manual_seed(seed + rows * dc)
    q = torch.randn(rows, 1, dc, generator=g).to(q_dt).cuda()
    C = torch.randn(256, dc, generator=g).cuda()
    W = (torch.randn(dc, d_out, generator=g) / dc ** 0.5).to(w_dt).cuda()
    return q, C, W, torch.arange(4, dtype=torch.int32).cuda()


@pytest.mark.parametrize("w_dt", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,dc,d_out", [(1, 8, 32), (31, 64, 96), (32, 72, 128), (33, 128, 1024), (96, 576, 4096),
                                           (128, 1024, 64), (129, 512, 64), (5, 320, 160)])
def test_projection_against_float64(rows, dc, d_out, w_dt):
    from intent_attention.triton_mla_decode import _projects, mla_decode_triton, mla_latent_context
    q, C, W, ids = _case(rows, dc, d_out, w_dt, torch.float32)
    ctx = mla_latent_context(q, C, ids, 64)
    assert _projects(ctx, W) == (rows <= 128)
    want = ctx.double() @ W.double()
    wide = torch.zeros(dc, d_out + 3, dtype=w_dt, device="cuda")
    wide[:, 1:d_out + 1] = W
    for w in (W, wide[:, 1:d_out + 1]):
        got = mla_decode_triton(q, C, w, ids, 64)
        # float32 sums of dc products: 1e-6 of the result's size
        assert float((got.double() - want).norm() / want.norm()) <= 1e-6
    for dt, half in ((torch.float16, 2 ** -11), (torch.bfloat16, 2 ** -8)):
        qh = q.to(dt)
        got = mla_decode_triton(qh, C, W, ids, 64)
        want = mla_latent_context(qh, C, ids, 64).double() @ W.double()
        assert got.dtype == dt and float((got.double() - want).abs().max()) <= float(want.abs().max()) * (half + 1e-5)


def test_what_stays_with_torch():
    from intent_attention.triton_mla_decode import _projects, mla_decode_triton
    q, C, W, ids = _case(4, 64, 64, torch.float32, torch.float32)
    plain = mla_decode_triton(q, C, W, ids, 64)
    Wg = W.clone().requires_grad_()
    out = mla_decode_triton(q, C, Wg, ids, 64)
    out.sum().backward()
    assert Wg.grad is not None and torch.allclose(out, plain, atol=1e-5)
    with torch.no_grad():
        assert torch.equal(mla_decode_triton(q, C, Wg, ids, 64), plain)
    t = W.t().contiguous().t()
    assert not _projects(q, t) and torch.allclose(mla_decode_triton(q, C, t, ids, 64), plain, atol=1e-5)
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(W, torch.ones_like(W))
        tangent = torch.autograd.forward_ad.unpack_dual(mla_decode_triton(q, C, dual, ids, 64)).tangent
        assert tangent is not None
    mapped = torch.func.vmap(lambda w: mla_decode_triton(q, C, w, ids, 64))(torch.stack([W, 2 * W]))
    assert torch.allclose(mapped[1], 2 * plain, atol=1e-5)
    with torch.autocast("cuda", dtype=torch.float16):
        assert not _projects(q, W)
