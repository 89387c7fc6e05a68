"""Host checks, no GPU: the module's products of a batch with a weight run over rows, never as a batched product over the
weight's expanded transpose (a bf16 form that has faulted on the GPU).  The operators that each call makes are recorded on
the CPU, with rows that are not evenly spaced: slices of longer sequences, transposes, one sequence of a larger buffer.  And the weights that a backward through operators sees."""
import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from transformer_amd import MLA, ModelArgs, training


class _Record(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.names.append(func.name())
        return func(*args, **(kwargs or {}))


def _uneven(K, dtype):
    g = torch.Generator().manual_seed(1)
    r = lambda *s: torch.randn(*s, generator=g).to(dtype)
    return [r(3, 7, K)[:, 1:6], r(5, 3, K).transpose(0, 1), r(4, 9, K)[1:2, :5], r(1, 1, K).expand(3, 5, K)]


@pytest.mark.parametrize("case", range(4))
def test_training_linear_forward_and_backward_have_no_batched_product(case):
    w = torch.nn.Parameter(torch.randn(24, 16, generator=torch.Generator().manual_seed(2)))
    x, dy = _uneven(16, torch.float32)[case].requires_grad_(True), _uneven(24, torch.float32)[case]
    with _Record() as rec:
        y = training.linear(x, w)
        got = torch.autograd.grad(y, (x, w), dy)
    assert not any("bmm" in n for n in rec.names), rec.names
    want = torch.autograd.grad(torch.nn.functional.linear(x, w), (x, w), dy)
    got += torch.autograd.grad(training.linear(x, w), (x, w), dy)  # without the mode: the plain backward
    for a, b in zip(got, want + want):
        torch.testing.assert_close(a, b)
    y = training.linear(x, w)
    y.add_(1)  # as torch's own output
    y.backward(dy)


@pytest.mark.parametrize("case", range(4))
def test_down_projections_without_gradients_have_no_batched_product(case):
    m = MLA(ModelArgs(d_model=256, n_heads=2, d_latent=128, q_lora_rank=128, max_seq_len=64)).to(torch.bfloat16)
    x = _uneven(256, torch.bfloat16)[case]
    with torch.no_grad(), _Record() as rec:
        y = m._down_all(x)
    assert any("mm" in n for n in rec.names) and not any("bmm" in n for n in rec.names), rec.names
    assert torch.equal(y, torch.nn.functional.linear(x.contiguous().clone(), m._down_w))


def test_operator_backward_sees_the_weights_of_the_forward():
    # weights written between forward and backward (a step with a retained graph): create_graph and a batch of gradients
    # use the forward's values, as the plain backward does, and a weight that is itself saved raises, as under torch's layer
    g = torch.Generator().manual_seed(4)
    ws = [torch.nn.Parameter(torch.randn(n, 16, generator=g)) for n in (8, 24)]
    x = torch.randn(2, 5, 16, generator=g).requires_grad_(True)
    dy = torch.randn(2, 5, 32, generator=g)
    leaves = [x, *ws]
    y = training.linear(x, *ws)
    want = torch.autograd.grad(y, leaves, dy, retain_graph=True)
    twice = [t.detach().clone() for t in _second(y, x, ws, dy)]
    with torch.no_grad():
        for w in ws:
            w.mul_(3)
    for got in (torch.autograd.grad(y, leaves, dy, retain_graph=True),
                torch.autograd.grad(y, leaves, dy, create_graph=True),
                [t[0] for t in torch.autograd.grad(y, leaves, dy[None], is_grads_batched=True, retain_graph=True)]):
        for a, b in zip(got, want):
            torch.testing.assert_close(a, b)
    for a, b in zip(_second(y, x, ws, dy), twice):
        torch.testing.assert_close(a, b)
    y = training.linear(x, ws[0])  # alone and in x's dtype: the weight itself is what is saved
    with torch.no_grad():
        ws[0].mul_(3)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        torch.autograd.grad(y, leaves[:2], dy[..., :8])


def _second(y, x, ws, dy):
    (gx,) = torch.autograd.grad(y, [x], dy, create_graph=True)
    return torch.autograd.grad(gx.square().sum(), ws)
