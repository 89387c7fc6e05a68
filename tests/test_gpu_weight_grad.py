"""mla_weight_grad (dW = dY^T X) and the training branch's linear layers built on it."""
import pytest
import torch

from tests import plans

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("out_fp32", [True, False])
@pytest.mark.parametrize("M,N,K,pad,narrow,S", [  # narrow, S: the tile and the token segments that the sizes take
    (1, 8, 8, 0, 1, 1),             # one token, one 16-byte chunk
    (31, 264, 136, 0, 1, 1),        # a ragged only stage, past one tile both ways
    (32, 256, 128, 8, 1, 1),        # one full stage, strided rows
    (33, 256, 256, 0, 1, 1),        # a one-token tail
    (97, 1000, 392, 24, 1, 1),      # four stages (the ring's depth) with a tail
    (160, 256, 256, 0, 1, 1),       # five stages: one through the steady loop
    (1000, 2624, 2048, 0, 1, 1),    # one segment, 176 narrow tiles
    (4100, 384, 1792, 16, 1, 9),    # many segments, the last one ragged
    (12288, 896, 384, 0, 1, 21),    # the segments' partials read eight at a time, and a remainder
    (33, 1800, 4104, 0, 0, 1),      # wide tiles, ragged both ways, a one-token tail
    (97, 1800, 4104, 16, 0, 1),     # wide tiles, four stages with a tail
    (129, 1800, 4104, 0, 0, 1),     # wide tiles, five stages
    (3001, 2056, 1800, 8, 0, 3),    # wide tiles in segments, ragged both ways, the last one shorter with a tail
    (6150, 2600, 2056, 0, 0, 2),    # the same, six tokens in the last stage
])
def test_weight_grad_matches_fp64(M, N, K, pad, narrow, S, out_fp32):
    plan = plans.weight_grad(M, N, K)
    assert (plan.narrow, plan.S) == (narrow, S), plan
    from transformer_amd import kernels
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    by = torch.randn(M, N + 2 * pad, generator=g, device="cuda").bfloat16()
    bx = torch.randn(M, K + 2 * pad, generator=g, device="cuda").bfloat16()
    dy, x = by[:, pad:pad + N], bx[:, pad:pad + K]
    dw = kernels.weight_grad(dy, x, out_fp32)
    ref = dy.double().t().contiguous() @ x.double().contiguous()
    # fp32 sums of M exact products: at most M 2^-24 of the sum of magnitudes; then one rounding to bf16
    mag = dy.double().abs().t().contiguous() @ x.double().abs().contiguous()
    bound = mag * (M + 8) * 2.0 ** -24
    if not out_fp32:
        bound = bound + (ref.abs() + bound) * 2.0 ** -8
    assert dw.dtype == (torch.float32 if out_fp32 else torch.bfloat16) and dw.shape == (N, K)
    assert ((dw.double() - ref).abs() <= bound).all()
    assert torch.equal(dw, kernels.weight_grad(dy, x, out_fp32)), "not bitwise reproducible"


def test_weight_grad_keeps_infinities_to_their_rows_and_the_padding_out():
    # 37 tokens: the stage's rows past the end and the columns past N and K hold NaN in memory
    from transformer_amd import kernels
    by = torch.full((64, 64), float("nan"), device="cuda").bfloat16()
    bx = torch.full((64, 64), float("nan"), device="cuda").bfloat16()
    by[:37, :24], bx[:37, :40] = 1, 1
    by[36, 3], bx[5, 7] = float("inf"), float("-inf")
    dw = kernels.weight_grad(by[:37, :24], bx[:37, :40], True).cpu()
    ref = torch.full((24, 40), 37.0)
    ref[3, :], ref[:, 7] = float("inf"), float("-inf")
    ref[3, 7] = float("nan")
    assert torch.equal(torch.nan_to_num(dw, nan=123.0), torch.nan_to_num(ref, nan=123.0))


def test_weight_grad_rejects_what_it_does_not_take():
    from transformer_amd import kernels
    z = lambda *s, dt=torch.bfloat16: torch.zeros(*s, dtype=dt, device="cuda")
    for dy, x, err in ((z(4, 12), z(4, 8), ValueError), (z(4, 8), z(4, 20), ValueError), (z(4, 8), z(5, 8), ValueError),
                       (z(0, 8), z(0, 8), ValueError), (z(4, 8, dt=torch.float32), z(4, 8), TypeError)):
        with pytest.raises(err):
            kernels.weight_grad(dy, x)


@pytest.mark.parametrize("amp", [True, False])
@pytest.mark.parametrize("frozen", [(), ("q_up", "kv_down"), ("q_down", "qk_rope", "kv_down"), ("k_up",)])
@pytest.mark.parametrize("shared", [False, True])
def test_module_gradients_equal_torch_layers(monkeypatch, amp, frozen, shared):
    """The training branch's linear layers against the same module on torch's own (plain_call false: what tracing, a mode
    or a transform makes it take), for fp32 weights under autocast and bf16 weights, with frozen weights: each gradient within bf16's rounding."""
    from transformer_amd import MLA, ModelArgs, training
    g = torch.Generator(device="cuda").manual_seed(3)
    with torch.device("cuda"):
        m = MLA(ModelArgs.mla_baseline(max_seq_len=256) if shared else ModelArgs(max_seq_len=256))
    for p in m.parameters():
        p.data.copy_(torch.randn(p.shape, generator=g, device="cuda") * 0.02)
    m = m if amp else m.to(torch.bfloat16)
    for n in frozen:
        m._modules[n].weight.requires_grad_(False)
    x0 = torch.randn(2, 150, m.d_model, generator=g, device="cuda").to(torch.bfloat16)
    dy = torch.randn(2, 150, m.d_model, generator=g, device="cuda").to(torch.bfloat16)

    def run():
        m.zero_grad(set_to_none=True)
        x = x0.clone().requires_grad_(True)
        with torch.autocast("cuda", dtype=torch.bfloat16, enabled=amp):
            y, _ = m(x)
        y.backward(dy)
        return [y.detach(), x.grad] + [p.grad for p in m.parameters()]

    calls = []
    real = training.linear
    monkeypatch.setattr(training, "linear", lambda *a, **k: calls.append(1) or real(*a, **k))
    ours = run()
    assert calls
    monkeypatch.setattr(training, "plain_call", lambda *t: False)
    n = len(calls)
    theirs = run()
    assert len(calls) == n
    for a, b in zip(ours, theirs):
        assert (a is None) == (b is None)
        if a is not None:
            assert a.dtype == b.dtype and a.shape == b.shape
            assert (a.double() - b.double()).norm() <= 1e-2 * b.double().norm()


def _small(**over):
    from transformer_amd import MLA, ModelArgs
    torch.manual_seed(5)
    with torch.device("cuda"):
        return MLA(ModelArgs(d_model=256, n_heads=2, d_latent=128, q_lora_rank=128, max_seq_len=128, **over)).to(
            torch.bfloat16)


def test_attention_function_under_saved_tensor_hooks_checkpoint_and_create_graph():
    """What autograd offers around the training branch works as around the operators: saved-tensor hooks, activation
    checkpointing, gradients through o_proj's own gradient, and the refusal to differentiate the attention twice."""
    m = _small()
    x = torch.randn(1, 70, 256, device="cuda").bfloat16().requires_grad_(True)
    dy = torch.randn_like(x)
    leaves = [x] + list(m.parameters())
    want = torch.autograd.grad(m(x)[0], leaves, dy)
    with torch.autograd.graph.save_on_cpu():
        got = torch.autograd.grad(m(x)[0], leaves, dy)
    assert all(torch.equal(a, b) for a, b in zip(want, got))
    y = torch.utils.checkpoint.checkpoint(lambda t: m(t)[0], x, use_reentrant=False)
    assert all(torch.equal(a, b) for a, b in zip(want, torch.autograd.grad(y, leaves, dy)))
    (g,) = torch.autograd.grad(m(x)[0], [m.o_proj.weight], dy, create_graph=True)
    second = torch.autograd.grad(g.float().square().sum(), [x, m.v_up.weight])
    assert all(torch.isfinite(t).all() and t.abs().max() > 0 for t in second)
    (g,) = torch.autograd.grad(m(x)[0], [x], dy, create_graph=True)
    with pytest.raises(RuntimeError):
        torch.autograd.grad(g.float().square().sum(), [x])


def test_linear_double_backward_and_hooked_layers():
    """create_graph through a layer alone (what torch's layer allows), and a hooked layer keeps its call."""
    from transformer_amd import training
    lin = torch.nn.Linear(64, 128, bias=False, device="cuda", dtype=torch.bfloat16)
    x = torch.randn(5, 64, device="cuda").bfloat16().requires_grad_(True)
    assert training.takes(lin, x)

    def penalty(f):
        gx, gw = torch.autograd.grad(f(x).square().sum(), (x, lin.weight), create_graph=True)
        return torch.autograd.grad(gx.float().square().sum() + gw.float().square().sum(), (x, lin.weight))

    for a, b in zip(penalty(lambda t: training.linear(t, lin.weight)), penalty(lin)):
        assert (a.double() - b.double()).norm() <= 2e-2 * b.double().norm()
    h = lin.register_forward_hook(lambda *a: None)
    assert not training.takes(lin, x)
    h.remove()
    with torch.no_grad():
        assert not training.takes(lin, x)


def test_batched_gradients_through_the_training_branch():
    """A batch of gradients in one call (is_grads_batched) gives what one call for each gives: norm, attention branch and
    o_proj, and a layer alone.  The two ways round at other places: three bf16 roundings of 2^-9, as many again inside."""
    from transformer_amd import RMSNorm, training
    m = _small()
    norm = RMSNorm(256).cuda()
    x = torch.randn(1, 70, 256, device="cuda").bfloat16().requires_grad_(True)
    dy = torch.randn(3, 1, 70, 256, device="cuda").bfloat16()
    leaves = [x, norm.weight] + list(m.parameters())
    lin = m.o_proj
    for y, at in ((m(norm(x))[0], leaves), (training.linear(x, lin.weight), [x, lin.weight])):
        got = torch.autograd.grad(y, at, dy, is_grads_batched=True, retain_graph=True)
        for i in range(3):
            for a, b in zip(got, torch.autograd.grad(y, at, dy[i], retain_graph=True)):
                assert (a[i].double() - b.double()).norm() <= 6 * 2.0 ** -9 * b.double().norm()


@pytest.mark.parametrize("weights", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B", [1, 2])
def test_expanded_gradients_and_overlapping_inputs(B, weights):
    """Gradients of sums (stride 0 over tokens, columns or both) and inputs whose rows repeat or overlap give what the
    same values as plain tensors give."""
    from transformer_amd import MLA, ModelArgs
    torch.manual_seed(8)
    with torch.device("cuda"):
        m = MLA(ModelArgs(d_model=256, n_heads=2, d_latent=128, q_lora_rank=128, max_seq_len=128))  # bf16 RoPE tables
    m = m.to(weights) if weights == torch.bfloat16 else m
    base = torch.randn(256 * 80, device="cuda").bfloat16()
    col = torch.randn(256, device="cuda").bfloat16()
    inputs = [base.as_strided((B, 37, 256), (128, 256, 1)), base.as_strided((B, 37, 256), (8, 128, 1)),
              base[:256].expand(B, 37, 256)]

    def grads(x, reduce):
        with torch.autocast("cuda", torch.bfloat16, enabled=weights == torch.float32):
            y = m(x)[0]
        return torch.autograd.grad(reduce(y), list(m.parameters()))

    for x in inputs:
        for reduce in (lambda y: y.float().sum(), lambda y: (y.sum((0, 1)) * col).sum(), lambda y: (y.sum(1) * col).sum(),
                       lambda y: y.sum()):
            got = grads(x, reduce)
            want = grads(x.clone(memory_format=torch.contiguous_format), reduce)
            assert all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("name", ["q_up", "k_up", "v_up", "o_proj"])
def test_replaced_layers_train_through_their_own_call(name):
    """A Sequential around a layer: the same gradients as the layer alone, each within bf16's rounding."""
    m = _small()
    x = torch.randn(2, 70, 256, device="cuda").bfloat16()
    dy = torch.randn_like(x)
    want = torch.autograd.grad(m(x)[0], list(m.parameters()), dy)
    calls = []
    m._modules[name] = torch.nn.Sequential(m._modules[name])
    m._modules[name].register_forward_hook(lambda *a: calls.append(1))
    for amp in (False, True):
        with torch.autocast("cuda", torch.bfloat16, enabled=amp):
            y = m(x)[0]
        for a, b in zip(torch.autograd.grad(y, list(m.parameters()), dy), want):
            assert (a.double() - b.double()).norm() <= 1e-2 * b.double().norm()
    assert len(calls) == 2


def test_undefined_gradients_give_zeros():
    """A consumer whose backward returns None: each operator's and the training branch's gradients are zeros."""
    import math
    from transformer_amd import RMSNorm, kernels, training

    class NoGrad(torch.autograd.Function):
        @staticmethod
        def forward(ctx, x):
            return x + 1

        @staticmethod
        def backward(ctx, g):
            return None

    r = lambda *s: torch.randn(*s, device="cuda").bfloat16().requires_grad_(True)
    m, norm = _small(), RMSNorm(256).cuda()
    x, qk = r(1, 40, 256), r(1, 40, 3, 64)
    q, k, v = r(1, 40, 2, 64), r(1, 40, 2, 64), r(1, 40, 2, 128)
    cos, sin = m.rope.cos_cached, m.rope.sin_cached
    scale = 1 / math.sqrt(128)
    calls = [(kernels.eager.rope(qk, cos, sin, 0, False), [qk]), (norm(x), [x, norm.weight]),
             (kernels.eager.prefill_fwd(q, r(1, 40, 2, 64), k, r(1, 40, 2, 64), v, scale, True, 0)[0], [q, k, v]),
             (kernels.eager.prefill_fwd_rope(q, r(1, 40, 2, 64), k, r(1, 40, 2, 64), v, cos, sin, scale, True, 0, 0,
                                             True)[0], [q, k, v]),
             (training.linear(x, m.o_proj.weight), [x, m.o_proj.weight]), (m(x)[0], [x] + list(m.parameters()))]
    for y, leaves in calls:
        assert all(g is not None and not g.any() for g in torch.autograd.grad(NoGrad.apply(y).sum(), leaves))


@pytest.mark.parametrize("tied", [False, True])
def test_operator_backward_of_the_attention_sees_the_weights_of_the_forward(tied):
    """fp32 weights under autocast, written between forward and backward: a batch of gradients and create_graph use the
    forward's values as the plain backward does (the two ways round at other places: as many roundings of 2^-9 as in
    test_batched_gradients_through_the_training_branch), also where k_up and v_up are one weight."""
    from transformer_amd import MLA, ModelArgs
    torch.manual_seed(9)
    with torch.device("cuda"):
        m = MLA(ModelArgs(d_model=256, n_heads=2, head_dim=192, d_latent=128, q_lora_rank=128, qk_nope_dim=128,
                          v_head_dim=128, max_seq_len=128))
    if tied:
        m.v_up.weight = m.k_up.weight
    x = torch.randn(1, 70, 256, device="cuda").requires_grad_(True)
    dy = torch.randn(1, 70, 256, device="cuda").bfloat16()
    leaves = [x] + list(m.parameters())
    with torch.autocast("cuda", torch.bfloat16):
        y = m(x)[0]
    want = torch.autograd.grad(y, leaves, dy, retain_graph=True)
    with torch.no_grad():
        for p in m.parameters():
            p.mul_(2)
    batched = [t[0] for t in torch.autograd.grad(y, leaves, dy[None], is_grads_batched=True, retain_graph=True)]
    for got in (torch.autograd.grad(y, leaves, dy, retain_graph=True), batched,
                torch.autograd.grad(y, leaves, dy, create_graph=True)):
        for a, b in zip(got, want):
            assert (a.double() - b.double()).norm() <= 6 * 2.0 ** -9 * b.double().norm()


@pytest.mark.parametrize("weights", [torch.bfloat16, torch.float32])
def test_compiled_training_gradients_equal_eager_ones_to_rounding(weights):
    """torch.compile keeps torch's layers and the registered operators, in one graph: each gradient within bf16's rounding
    of the eager branch's."""
    from contextlib import nullcontext
    from transformer_amd import MLA, ModelArgs
    torch.manual_seed(13)
    with torch.device("cuda"):
        m = MLA(ModelArgs(d_model=256, n_heads=2, d_latent=128, q_lora_rank=128, max_seq_len=128))  # bf16 RoPE tables
    m = m.to(weights) if weights == torch.bfloat16 else m
    x = torch.randn(2, 70, 256, device="cuda").to(weights).requires_grad_(True)
    dy = torch.randn(2, 70, 256, device="cuda").bfloat16()
    leaves = [x] + list(m.parameters())
    amp = nullcontext() if weights == torch.bfloat16 else torch.autocast("cuda", torch.bfloat16)
    torch._dynamo.reset()
    with amp:
        compiled = torch.compile(lambda t: m(t)[0], backend="eager", fullgraph=True)(x)
        eager = m(x)[0]
    for a, b in zip(torch.autograd.grad(compiled, leaves, dy), torch.autograd.grad(eager, leaves, dy)):
        assert a.dtype == b.dtype and (a.double() - b.double()).norm() <= 1e-2 * b.double().norm()
