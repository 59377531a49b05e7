"""ops/_native.py dispatch helpers: env_flag follows os.environ changes made at run time (monkeypatch.setenv, smoke()'s
LIPA_REFERENCE toggle), and fn_apply builds the same autograd graph as Function.apply."""
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.fx.experimental.proxy_tensor import make_fx

from llm_in_practise_amd.ops._native import eager, env_flag, fn_apply, force_reference
from llm_in_practise_amd.ops.loss import shift_labels


def test_env_flag_tracks_runtime_changes(monkeypatch):
    monkeypatch.delenv("LIPA_REFERENCE", raising=False)
    assert not force_reference() and not env_flag("LIPA_REFERENCE")
    monkeypatch.setenv("LIPA_REFERENCE", "1")
    assert force_reference()
    monkeypatch.setenv("LIPA_REFERENCE", "0")
    assert not force_reference()


class _Scale(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, w, k):
        ctx.save_for_backward(w)
        ctx.k = k
        return x * w * k

    @staticmethod
    def backward(ctx, g):
        (w,) = ctx.saved_tensors
        return g * w * ctx.k, None, None


def test_fn_apply_matches_function_apply():
    x = torch.randn(5, requires_grad=True)
    w = torch.randn(5)
    y1 = _Scale.apply(x, w, 3.0)
    g1, = torch.autograd.grad(y1.sum(), x)
    y2 = fn_apply(_Scale, x, w, 3.0)
    g2, = torch.autograd.grad(y2.sum(), x)
    assert torch.equal(y1, y2) and torch.equal(g1, g2)
    assert type(y2.grad_fn).__name__ == type(y1.grad_fn).__name__
    with torch.no_grad():
        assert fn_apply(_Scale, x, w, 2.0).grad_fn is None


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
