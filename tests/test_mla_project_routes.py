"""Which W_VO the MLA projection's kernel takes, on the host: a plain row-major one, and none for
which torch's product does more than multiply."""
import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from intent_attention.triton_mla_decode import _projects

CTX = torch.zeros(2, 1, 64)
W = torch.ones(64, 32)


def test_a_plain_w():
    assert _projects(CTX, W) and _projects(CTX, torch.nn.Parameter(W, requires_grad=False))
    assert not _projects(CTX, W.t().contiguous().t()) and not _projects(CTX, W.double())


@pytest.mark.parametrize("form", ["to_sparse", "to_sparse_csr", "to_sparse_csc"])
@pytest.mark.filterwarnings("ignore:Sparse")
def test_a_sparse_w_stays_with_torch(form):
    w = getattr(W, form)()
    assert not _projects(CTX, w)
    assert torch.equal(CTX @ w.float(), CTX @ W)          # which multiplies it


def test_a_product_that_is_recorded_stays_with_torch():
    """A trace, or a dispatch mode (a counter of operations, say), sees the product by W."""
    seen = []

    def project(w):
        seen.append(_projects(CTX, w))
        return CTX @ w.float()

    torch.jit.trace(project, (W,), check_trace=False)

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    with Mode():
        project(W)
    project(W)
    assert seen == [False, False, True]
