"""What semantic_block_attention attends to, on the host: the tokens its layout selects, whoever
selects them, and where it may read them in place. The attention itself is stood in for."""
import pytest
import torch

from intent_attention import BlockLayout, BlockPolicy, SemanticBlock, reference


@pytest.fixture
def calls(monkeypatch):
    """(form, token indices) of each attention call."""
    seen = []

    def in_place(q, k, v, causal, mask, positions, kv_index=None):
        seen.append(("in place", kv_index.tolist()))
        return torch.zeros_like(q)

    def gathered(q, k, v, causal=False, mask=None, original_kv_positions=None):
        assert k.shape[-2] == v.shape[-2] == original_kv_positions.shape[0]
        assert torch.equal(k[0, :, 0], original_kv_positions.float())
        seen.append(("gathered", original_kv_positions.tolist()))
        return torch.zeros_like(q)

    monkeypatch.setattr(reference, "require_device", lambda *t, what="": t[0].device)
    monkeypatch.setattr(reference, "_dense_attention", in_place)
    monkeypatch.setattr(reference, "dense_attention", gathered)
    return seen


def _qkv(tokens=40):
    k = torch.arange(tokens).float()[None, :, None].expand(2, tokens, 4).contiguous()
    return torch.zeros(2, 3, 4), k, k.clone()


def _layout(cls=BlockLayout, *bounds):
    return cls([SemanticBlock(f"b{i}", s, e, BlockPolicy.ALWAYS) for i, (s, e) in enumerate(bounds)])


def test_spans_are_read_in_place(calls):
    reference.semantic_block_attention(*_qkv(), _layout(BlockLayout, (0, 3), (7, 9)))
    assert calls == [("in place", [0, 1, 2, 7, 8])]


@pytest.mark.parametrize("bounds", [(0.0, 8.0), (0.5, 3.2), (0, 8.0)])
def test_bounds_that_are_not_whole_numbers_are_refused(calls, bounds):
    with pytest.raises(TypeError, match="integer"):
        reference.semantic_block_attention(*_qkv(), _layout(BlockLayout, bounds))
    assert not calls
