"""mla_paged_decode with few heads (csrc/mla_few.h): head counts around the 16 of a
workgroup, from one page to more than a wave's share, every latent shape, value offset
and page format, ragged lengths and splits, against the float64 oracle; and the
head counts either side of the rule that picks the form."""
import numpy as np
import pytest

from oracle import mla as M
from test_gpu_mla import SHAPES, _device_pools, _latent_case

pytestmark = pytest.mark.gpu

MIXES = {"fp16": {"FP16": .9, "SKIP": .1}, "codes": {"FP8": .45, "INT8": .45, "SKIP": .1},
         "all": {"FP16": .4, "FP8": .25, "INT8": .25, "SKIP": .1}}


@pytest.mark.parametrize("dqk,dv,voff", SHAPES, ids=[f"{a}x{b}+{c}" for a, b, c in SHAPES])
@pytest.mark.parametrize("mix", sorted(MIXES))
@pytest.mark.parametrize("heads,W,pps", [(1, 1, 0), (8, 5, 0), (16, 37, 0), (15, 70, 70), (17, 33, 9), (5, 140, 128)])
def test_few_heads_match_the_oracle(dqk, dv, voff, mix, heads, W, pps):
    import torch
    from intent_attention import mla_paged_decode
    dev = torch.device("cuda:0")
    q, pools, table, counts, tags = _latent_case(7 * dqk + heads + W, 2, heads, dqk, 160, W, MIXES[mix])
    valid = (counts * 16).astype(np.int32)
    valid[1] = max(1, valid[1] - 7)
    for dt in (torch.float16, torch.bfloat16, torch.float32):
        qt = torch.from_numpy(q).to(dev).to(dt)
        got = mla_paged_decode(qt, _device_pools(pools, dev), torch.from_numpy(table).to(dev),
                               torch.from_numpy(counts).to(dev), torch.from_numpy(tags).to(dev), v_dim=dv, v_offset=voff,
                               valid_tokens=torch.from_numpy(valid).to(dev), pages_per_split=pps, out_dtype=torch.float32)
        ref = M.mla_paged_decode_oracle(qt.float().cpu().numpy(), pools, table, counts, tags, v_dim=dv, v_offset=voff,
                                        valid_tokens=valid)
        err = np.abs(got.cpu().numpy() - ref).max()
        assert err <= 1e-2, (str(dt), f"max abs err {err:.3e}")     # the bar of the 128-head form's tests


@pytest.mark.parametrize("heads,batch,W", [(16, 3, 300), (17, 3, 300), (48, 1, 512), (128, 2, 256), (128, 2, 257), (96, 3, 64)])
def test_either_side_of_the_rule(heads, batch, W):
    import torch
    from intent_attention import mla_paged_decode
    dev = torch.device("cuda:0")
    for mix in ("fp16", "codes"):
        q, pools, table, counts, tags = _latent_case(heads + W, batch, heads, 576, 600, W, MIXES[mix])
        got = mla_paged_decode(torch.from_numpy(q).to(dev), _device_pools(pools, dev), torch.from_numpy(table).to(dev),
                               torch.from_numpy(counts).to(dev), torch.from_numpy(tags).to(dev), v_dim=512)
        ref = M.mla_paged_decode_oracle(q, pools, table, counts, tags, v_dim=512)
        assert np.abs(got.float().cpu().numpy() - ref).max() <= 1e-2
