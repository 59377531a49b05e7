"""ops/_native.py's eager(): tensors that a kernel cannot read, and calls that something records, keep torch's operations."""
import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.fx.experimental.proxy_tensor import make_fx

from llm_in_practise_amd.ops._native import eager
from llm_in_practise_amd.ops.gemm import _base_gemm
from llm_in_practise_amd.ops.loss import shift_labels
from llm_in_practise_amd.ops.mlp import skinny_swiglu


def _legacy_rows(seen):
    """``seen`` of the batched gradient that a backward gets from ``is_grads_batched``."""
    class Look(torch.autograd.Function):
        @staticmethod
        def forward(ctx, x):
            return x * 1

        @staticmethod
        def backward(ctx, g):
            seen(g)
            return g
    x = torch.ones(3, requires_grad=True)
    torch.autograd.grad(Look.apply(x), x, torch.eye(3), is_grads_batched=True)


def test_eager_means_plain_tensors_and_nothing_recording():
    x, got = torch.ones(3), []

    def seen(t):
        got.append(eager(t))
        return t * 1
    assert eager(x, None, torch.nn.Parameter(x)) and not eager(x, x.as_subclass(type("Own", (torch.Tensor,), {})))
    seen(x)
    assert got.pop()
    _legacy_rows(seen)
    torch.func.vmap(seen)(torch.ones(2, 3))
    torch.func.grad(lambda t: seen(t).sum())(x)
    make_fx(seen)(x)
    torch.jit.trace(seen, x, check_trace=False)
    with torch.autograd.forward_ad.dual_level():
        seen(torch.autograd.forward_ad.make_dual(x, x))
    with FakeTensorMode():
        seen(torch.ones(3))
    assert len(got) == 7 and not any(got)
    assert eager(x)


def test_shift_labels_of_tensors_without_memory():
    """Fake tensors of a GPU, and a trace of them: torch's operations, nothing that reads an address."""
    with FakeTensorMode():
        labels = torch.zeros(2, 8, dtype=torch.int64, device="cuda")
        out = shift_labels(labels)
        assert out.shape == (2, 8) and out.device.type == "cuda"
        nodes = [n.target for n in make_fx(lambda t: shift_labels(t))(labels).graph.nodes if n.op == "call_function"]
        assert len(nodes) > 1


@pytest.mark.parametrize("M,N,K", [(12, 1024, 12288), (17, 1024, 1024), (64, 4096, 4096), (32, 2560, 9728)])
def test_narrow_products_of_tensors_without_memory(M, N, K):
    """Fake rows and weights of a GPU keep the library's product, traced or not, and no gated launch."""
    with FakeTensorMode():
        x, w = (torch.zeros(s, dtype=torch.bfloat16, device="cuda") for s in ((M, K), (N, K)))
        assert _base_gemm(x, w).shape == (M, N)
        nodes = [n.target for n in make_fx(lambda a, b: _base_gemm(a, b))(x, w).graph.nodes if n.op == "call_function"]
        assert torch.ops.aten.mm.default in nodes
        if M > 16:
            assert skinny_swiglu(x[:, :1024], torch.zeros(6144, 1024, dtype=torch.bfloat16, device="cuda")) is None
