"""Which dense calls take one launch (the library's workspace rule, no device needed): a
workspace of 0 bytes is the row form on its own, NO_SCRATCH the matrix form on its own,
more is a call whose keys are split or whose key tiles are flagged, with a kernel behind it."""
import pytest

from intent_attention import _native as N


def _workspace(dtype, batch, q_len, kv_len, dim, causal=0, mask=False):
    a = N.DenseAttentionArgs()
    a.batch, a.q_len, a.kv_len, a.head_dim, a.v_dim, a.dtype = batch, q_len, kv_len, dim, dim, dtype
    base = 1 << 20
    a.q = a.k = a.v = a.out = base
    a.q_stride_b, a.q_stride_t, a.k_stride_b, a.k_stride_t = q_len * dim, dim, kv_len * dim, dim
    a.v_stride_b, a.v_stride_t, a.out_stride_b, a.out_stride_t = kv_len * dim, dim, q_len * dim, dim
    a.causal, a.sm_scale = causal, dim ** -0.5
    if mask:
        a.mask, a.mask_dtype, a.mask_stride_q, a.mask_stride_k = base, dtype, kv_len, 1
    return N.dense_attention_workspace(a)


ROW, ONE, MORE = "row form alone", "matrix form alone", "two kernels"


def _kind(n):
    return ROW if n == 0 else ONE if n == N.DENSE_NO_SCRATCH else MORE


@pytest.mark.parametrize("dtype", [N.DTYPE_F16, N.DTYPE_BF16])
@pytest.mark.parametrize("shape,kw,want", [
    ((16, 32, 256, 64), {}, ONE), ((32, 8, 600, 64), {}, ONE), ((16, 16, 512, 128), {}, ONE), ((16, 16, 513, 128), {}, MORE),
    ((16, 16, 333, 80), dict(mask=True), ONE), ((32, 2, 1024, 64), dict(mask=True), MORE), ((2, 128, 257, 64), {}, ONE),
    ((8, 64, 64, 128), dict(causal=1), ONE), ((32, 2048, 2048, 128), dict(causal=1), MORE), ((8, 1, 64, 64), {}, ROW),
    ((1000, 130, 100, 64), {}, ONE), ((70, 100, 190, 192), {}, MORE)])
def test_short_16_bit_calls_are_one_kernel(dtype, shape, kw, want):
    assert _kind(_workspace(dtype, *shape, **kw)) == want


@pytest.mark.parametrize("shape,kw,want", [
    ((16, 32, 256, 64), {}, ONE), ((16, 16, 400, 64), {}, ROW), ((16, 32, 400, 64), {}, MORE),
    ((300, 3, 128, 128), {}, ROW), ((8, 128, 200, 128), {}, MORE), ((48, 1, 2048, 128), {}, MORE), ((16, 3, 2048, 128), {}, MORE),
    ((300, 40, 64, 64), {}, ONE), ((300, 200, 2000, 128), {}, ONE), ((300, 200, 2000, 128), dict(causal=1), MORE)])
def test_float32_calls(shape, kw, want):
    assert _kind(_workspace(N.DTYPE_F32, *shape, **kw)) == want
