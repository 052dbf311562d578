"""Host arguments of the device entry points under torch's own settings: what plain tensors
and lists did before, they do under a default device too."""
import pytest
import torch

from intent_attention import page_tables as P


@pytest.mark.parametrize("arrays", [[("a", [3, 1, 2]), ("b", [])], [("a", [2 ** 31 - 1])]])
def test_upload_under_a_default_device(arrays):
    cpu = torch.device("cpu")
    plain = P._upload(arrays, cpu)
    with torch.device("meta"):                 # as torch.set_default_device("cuda") in a program
        got = P._upload(arrays, cpu)
    for x, y in zip(got, plain):
        assert x.device == cpu and x.dtype == torch.int32 and torch.equal(x, y)
