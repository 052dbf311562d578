"""The split plan of the paged MLA decode (no device needed): which form a call takes, read off the
number of splits that its workspace holds."""
import ctypes

import pytest

from intent_attention import _native as N


def _splits(batch, heads, width, fp16, codes, dqk=576, dv=512):
    a = N.MlaDecodeArgs()
    a.batch, a.num_heads, a.qk_dim, a.v_dim, a.page_size, a.table_width, a.num_pages = batch, heads, dqk, dv, 16, width, 4096
    base = 1 << 20
    a.q = a.out = a.page_table = a.page_counts = a.page_tags = base
    a.q_stride_b, a.q_stride_h, a.out_stride_b, a.out_stride_h = heads * dqk, dqk, heads * dv, dv
    for t in range(8):
        a.tag_map[t] = N.TAG_SKIP
    if fp16:
        a.tag_map[0], a.c_fp16 = N.TAG_FP16, base
    if codes:
        a.tag_map[1], a.c_int8, a.c_int8_scale = N.TAG_INT8, base, base
    a.sm_scale = 1.0
    n = ctypes.c_size_t(0)
    N.check(N.load().iak_mla_decode_workspace(ctypes.byref(a), ctypes.byref(n)))
    return max(1, round(n.value / (batch * heads * (dv + 2) * 4)))


def _many(batch, width):    # one workgroup per (sequence, split): 256 of them
    chunk = -(-width // (-(-256 // batch)))
    return -(-width // chunk)


def _few(batch, heads, width):   # one per 16 heads, 256 at most, four pages or more each
    want = max(1, 256 // (batch * -(-heads // 16)))
    chunk = max(4, -(-width // want))
    return -(-width // chunk)


@pytest.mark.parametrize("batch,heads,width,fp16,codes,few", [
    (8, 16, 64, True, False, True), (8, 16, 64, True, True, True), (8, 16, 64, False, True, False),
    (8, 8, 64, False, True, True), (2, 64, 256, True, True, True), (2, 64, 256, False, True, True),
    (2, 64, 257, False, True, False), (2, 48, 512, False, True, False), (2, 64, 512, True, False, True),
    (2, 64, 513, True, False, False), (1, 32, 1024, False, True, False), (1, 32, 2048, True, True, True),
    (3, 17, 100, True, False, False)])
def test_form_by_heads_pages_and_pools(batch, heads, width, fp16, codes, few):
    got = _splits(batch, heads, width, fp16, codes)
    assert _few(batch, heads, width) != _many(batch, width)
    assert got == (_few(batch, heads, width) if few else _many(batch, width))
