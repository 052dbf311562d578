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


class _EveryThird(BlockLayout):
    def selected_token_indices(self):
        return super().selected_token_indices()[::3]


class _Outside(BlockLayout):
    def validate(self, total_tokens):
        pass


def test_a_layout_that_selects_its_own_tokens(calls):
    reference.semantic_block_attention(*_qkv(), _layout(_EveryThird, (0, 3), (7, 12)))
    one = _layout(BlockLayout, (0, 30))
    one.selected_token_indices = lambda: [4, 2, 2]
    _, debug = reference.semantic_block_attention(*_qkv(), one, return_debug=True)
    assert calls == [("gathered", [0, 7, 10]), ("gathered", [4, 2, 2])] and debug["selected_kv_tokens"] == 3
    one.selected_token_indices = lambda: []
    out = reference.semantic_block_attention(*_qkv(), one)
    assert len(calls) == 2 and not out.any()


@pytest.mark.parametrize("bounds", [(30, 50), (-2, 5)])
def test_tokens_outside_are_not_read_in_place(calls, bounds):
    """Without BlockLayout's validation the gather is what checks the tokens (index_select raises)."""
    with pytest.raises((IndexError, RuntimeError)):
        reference.semantic_block_attention(*_qkv(), _layout(_Outside, bounds))
    assert not calls
