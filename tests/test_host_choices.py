"""Host-side choices that need no GPU: when the decode step's few-row products go to
linear_rows (transformer.py:208-213, :252-254, :300 at T == 1), when a chunk over a cache takes
the absorbed kernel (:249-291 with T > 1), and the backward's workspace falling back to the
recompute path when the stored-dS workspace cannot be allocated."""
from types import SimpleNamespace

import ctypes

import pytest
import torch


def test_rows_path_needs_autograd_off_few_rows_bf16_and_fitting_dims():
    from transformer_amd import MLA, ModelArgs
    m = MLA(ModelArgs.mla_baseline(max_seq_len=64)).to(torch.bfloat16)
    x = torch.zeros(32, 1, m.d_model, dtype=torch.bfloat16)
    assert not m._rows_path(x)  # autograd on: the training path keeps nn.Linear
    with torch.no_grad():
        assert m._rows_path(x)
        assert m._rows_path(torch.zeros(64, 1, m.d_model, dtype=torch.bfloat16))
        assert not m._rows_path(torch.zeros(65, 1, m.d_model, dtype=torch.bfloat16))
        assert not m.float()._rows_path(x.float())  # fp32 arithmetic outside autocast
    # dims the kernel does not take (d_model 64: K not a multiple of 128) stay on nn.Linear
    small = MLA(SimpleNamespace(d_model=64, n_heads=4, head_dim=128, d_latent=64, q_lora_rank=64,
                                max_seq_len=64)).to(torch.bfloat16)
    with torch.no_grad():
        assert not small._rows_path(torch.zeros(1, 1, 64, dtype=torch.bfloat16))


def test_absorbed_chunk_choice():
    # benchmark dims (d_latent 512, nope 128 + rope 64, v 128, shared k_rope): the absorbed kernel
    # costs 1088 multiply-adds per key, head and query against 131072 per key and head to
    # up-project the cache plus 320 per query: short chunks take it, long ones do not
    from transformer_amd import MLA, ModelArgs
    import transformer_amd.mla as M
    m = MLA(ModelArgs.mla_baseline(max_seq_len=64))
    shared = torch.zeros(2, 1, 8, 64)
    with torch.no_grad():
        assert m._absorbed_prefill_ok(2, shared) and m._absorbed_prefill_ok(64, shared)
        assert m._absorbed_prefill_ok(119, shared) and not m._absorbed_prefill_ok(120, shared)
        assert not m._absorbed_prefill_ok(64, torch.zeros(2, 16, 8, 64))  # per-head k_rope
    assert not m._absorbed_prefill_ok(64, shared)  # autograd on: the path with a backward
    saved = M.ABSORBED_PREFILL
    try:
        M.ABSORBED_PREFILL = False
        with torch.no_grad():
            assert not m._absorbed_prefill_ok(64, shared)
    finally:
        M.ABSORBED_PREFILL = saved


def test_rows_fit_limits():
    from transformer_amd import kernels
    assert kernels.rows_fit(128, 4) and kernels.rows_fit(4096, 2624)
    assert not kernels.rows_fit(64, 4) and not kernels.rows_fit(4224, 4) and not kernels.rows_fit(2048, 6)
    assert not kernels.rows_fit(0, 4)


def test_backward_workspace_falls_back_when_the_stored_ds_allocation_fails(monkeypatch):
    from transformer_amd import _lib, kernels
    a = _lib.PrefillBwdArgs()
    a.B, a.H, a.Tq, a.Tk, a.d_nope, a.d_rope, a.d_v, a.causal = 4, 16, 4096, 4096, 128, 64, 128, 1
    full = int(_lib.entry("mla_prefill_bwd_workspace_bytes")(ctypes.byref(a)))
    small = int(_lib.entry("mla_prefill_bwd_workspace_min_bytes")(ctypes.byref(a)))
    assert full > small > 0
    asked = []

    def alloc(nbytes, dev):
        asked.append(nbytes)
        if nbytes > small:
            raise torch.OutOfMemoryError("mocked")
        return torch.empty(max(nbytes, 1), dtype=torch.uint8)

    monkeypatch.setattr(kernels, "_alloc_workspace", alloc)
    ws, nbytes = kernels._bwd_workspace(a, torch.device("cpu"))
    assert asked == [full, small] and nbytes == small and ws.numel() == small
    monkeypatch.setattr(kernels, "BWD_STORED_DS", False)
    asked.clear()
    assert kernels._bwd_workspace(a, torch.device("cpu"))[1] == small and asked == [small]


def test_split_column_product_equals_the_one_product():
    # the down-projection's two-product form, on the host: the same values as x @ W^T, written
    # into the columns of one output
    import transformer_amd.mla as M
    g = torch.Generator().manual_seed(3)
    x = torch.randn(3, 5, 64, generator=g, dtype=torch.float64)
    W = torch.randn(300, 64, generator=g, dtype=torch.float64)
    y = M._linear_split_cols(x, W)
    assert y.shape == (3, 5, 300)
    torch.testing.assert_close(y, x @ W.t(), rtol=1e-12, atol=1e-12)
    assert M._split_pays(24576, 2624) and not M._split_pays(24576, 2560) and not M._split_pays(512, 2624)
    assert not M._split_pays(4096, 200)  # below one 256-column block


def test_eager_ops_take_the_registered_operator_when_it_is_needed():
    # the module layer calls the op bodies directly only when the dispatcher adds nothing: no
    # tracing, dispatch mode, functorch transform, subclass, off-GPU tensor or needed gradient
    from torch._subclasses.fake_tensor import FakeTensorMode
    from transformer_amd import kernels
    need = kernels.dispatcher_needed
    assert not need(()) and not need((1, 2.0, None))
    assert need((torch.zeros(2),))  # a CPU tensor takes the operator (which raises: no CPU path)
    assert need((torch.zeros(2, device="meta"),))  # meta tensors take the fake kernels
    with FakeTensorMode():
        assert need(())
    seen = []
    torch.func.vmap(lambda t: seen.append(need(())) or t)(torch.zeros(3, 2))
    assert seen == [True]
    compiled = torch.compile(lambda t: t + (1 if need(()) else -1), backend="eager", fullgraph=True)
    assert compiled(torch.zeros(1)).item() == 1
    assert all(hasattr(torch.ops.mla_mi355x, n) for n in vars(kernels.eager)) and len(vars(kernels.eager)) == 17
    with pytest.raises(RuntimeError, match="ROCm GPU"):
        kernels.eager.rope(torch.zeros(1, 2, 1, 64, dtype=torch.bfloat16), torch.zeros(4, 32, dtype=torch.bfloat16),
                           torch.zeros(4, 32, dtype=torch.bfloat16), 0, False)


def test_backward_stored_ds_workspace_counts_the_visible_blocks():
    # the stored-dS part of the backward's workspace (its size minus the recompute path's, rounded to
    # 256 bytes) is 2 KiB per 32 x 32 block that the dK/dV pass stores: query block i stores key block j
    # when the block's last query row sees the block's first key (j < ceil(Tk / 32); causal:
    # 32 j <= 32 i + 31 + q_offset), counted here by enumeration; above 8 GiB there is no dS part
    import random
    from transformer_amd import _lib

    def sizes(B, H, Tq, Tk, q_offset, causal):
        a = _lib.PrefillBwdArgs()
        a.B, a.H, a.Tq, a.Tk, a.d_nope, a.d_rope, a.d_v = B, H, Tq, Tk, 128, 64, 128
        a.q_offset, a.causal = q_offset, int(causal)
        full = int(_lib.entry("mla_prefill_bwd_workspace_bytes")(ctypes.byref(a)))
        small = int(_lib.entry("mla_prefill_bwd_workspace_min_bytes")(ctypes.byref(a)))
        return full, small

    def enumerated(B, H, Tq, Tk, q_offset, causal):
        nqb, nkb = (Tq + 31) // 32, (Tk + 31) // 32
        n = sum(1 for i in range(nqb) for j in range(nkb) if not causal or 32 * j <= 32 * i + 31 + q_offset)
        return B * H * n * 2048

    rng = random.Random(5)
    cases = [(1, 1, 32, 32, 0, True), (1, 1, 33, 33, 0, True), (2, 3, 100, 250, 150, True), (1, 2, 64, 31, 0, True),
             (1, 1, 70, 70, 31, True), (1, 1, 70, 70, 32, True), (1, 1, 70, 70, 33, True), (1, 1, 40, 500, 1000, True),
             (3, 2, 77, 45, 0, False), (1, 16, 4096, 4096, 0, True)]
    cases += [(rng.randint(1, 3), rng.randint(1, 4), rng.randint(1, 400), rng.randint(1, 400), rng.choice([0, 0, 1, 31, 32,
              rng.randint(0, 500)]), rng.random() < 0.8) for _ in range(200)]
    for B, H, Tq, Tk, q_offset, causal in cases:
        full, small = sizes(B, H, Tq, Tk, q_offset, causal)
        assert full - ((small + 255) // 256 * 256) == enumerated(B, H, Tq, Tk, q_offset, causal), \
            (B, H, Tq, Tk, q_offset, causal)
    full, small = sizes(16, 16, 16384, 16384, 0, True)  # 17.2 GB of dS blocks: over the cap, recompute path
    assert full == small


def test_autograd_functions_stand_in_only_in_plain_eager_mode():
    # the eager calls' autograd.Functions (and the training branch's) give way to the registered operators wherever
    # something would see less: a trace, a mode, a transform, forward-mode, tensors that are not plain
    from torch._subclasses.fake_tensor import FakeTensorMode
    from torch.overrides import TorchFunctionMode
    from transformer_amd import kernels
    fits = kernels.function_fits
    assert fits(()) and fits((1, None)) and not fits((torch.zeros(2),)) and not fits((torch.zeros(2, device="meta"),))
    with FakeTensorMode():
        assert not fits(())

    class Mode(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    with Mode():
        assert not fits(())
    with torch.autograd.forward_ad.dual_level():
        assert not fits(())
    seen = []
    torch.func.grad(lambda t: (seen.append(fits(())), t.sum())[1])(torch.zeros(3))
    torch.jit.trace(lambda t: (seen.append(fits(())), t + 1)[1], torch.zeros(3), check_trace=False)
    assert seen and not any(seen)
    assert torch.compile(lambda t: t + (-1 if fits(()) else 1), backend="eager", fullgraph=True)(torch.zeros(1)).item() == 1


def test_training_layers_take_only_plain_linears():
    from transformer_amd import training
    lin = torch.nn.Linear(8, 8, bias=False)
    assert training.plain_linear(lin)
    assert not training.plain_linear(torch.nn.Linear(8, 8)) and not training.plain_linear(torch.nn.Identity())
    sub = type("Sub", (torch.nn.Linear,), {})(8, 8, bias=False)
    assert not training.plain_linear(sub)
    for hook in (lin.register_forward_pre_hook, lin.register_forward_hook, lin.register_full_backward_hook):
        h = hook(lambda *a: None)
        assert not training.plain_linear(lin)
        h.remove()
    h = torch.nn.modules.module.register_module_forward_hook(lambda *a: None)
    assert not training.plain_linear(lin)
    h.remove()
    assert training.plain_linear(lin)
    torch.nn.utils.parametrizations.weight_norm(lin)
    assert not training.plain_linear(lin)


def test_rows_path_takes_the_projections_where_only_the_absorption_does_not_fit():
    # the reference's default dims: W_UK's K = 64 is outside linear_rows, the projections are inside
    from transformer_amd import MLA, ModelArgs
    m = MLA(ModelArgs(max_seq_len=64)).to(torch.bfloat16)
    x = torch.zeros(4, 1, m.d_model, dtype=torch.bfloat16)
    with torch.no_grad():
        assert m._rows_proj_ok() and not m._rows_dims_ok() and m._rows_path(x)
        assert not m._rows_path(torch.zeros(65, 1, m.d_model, dtype=torch.bfloat16))


@pytest.mark.parametrize("baseline", [True, False])
@pytest.mark.parametrize("layer", ["q_up", "o_proj"])
def test_rows_path_calls_layers_that_are_more_than_a_product(layer, baseline, monkeypatch):
    # a hook, a wrapper that passes the weight on (an adapter), a parametrization (a fresh weight on each access), a layer
    # of another kind: the few-row products read weights, so they give way to the layers' own calls
    from transformer_amd import MLA, ModelArgs
    import torch.nn as nn
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)  # (asks a GPU)

    class Adapter(nn.Module):
        def __init__(self, inner):
            super().__init__()
            self.inner = inner

        @property
        def weight(self):
            return self.inner.weight

        def forward(self, x):
            return self.inner(x) * 2

    def make():
        m = MLA(ModelArgs.mla_baseline(max_seq_len=64) if baseline else ModelArgs(max_seq_len=64)).to(torch.bfloat16)
        return m, m._modules[layer]

    def hooked(m, lin):
        lin.register_forward_hook(lambda *a: None)

    def wrapped(m, lin):
        m._modules[layer] = Adapter(lin)

    def several(m, lin):
        m._modules[layer] = nn.Sequential(lin)

    def parametrized(m, lin):
        nn.utils.parametrize.register_parametrization(lin, "weight", nn.Identity())

    with torch.no_grad():
        for change in (None, hooked, wrapped, several, parametrized):
            m, lin = make()
            x = torch.zeros(40, 1, m.d_model, dtype=torch.bfloat16)
            if change:
                change(m, lin)
            assert m._rows_path(x) == (change is None), change
            assert m._auto_graph_ok(x) == (change is None), change


def test_rows_path_keeps_no_copies_of_fp32_weights_where_the_layers_ran(monkeypatch):
    # fp32 weights under bf16 autocast: the reference's default dims keep q_up and o_proj as layers, and no layout reads a
    # kept copy in a capture; bf16 weights are read as they are
    from transformer_amd import MLA, ModelArgs
    capturing = [False]
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capturing[0])
    amp = [True]
    monkeypatch.setattr(torch, "is_autocast_enabled", lambda *a: amp[0])  # (no GPU: torch turns autocast off)
    monkeypatch.setattr(torch, "get_autocast_dtype", lambda *a: torch.bfloat16)
    for baseline in (True, False):
        m = MLA(ModelArgs.mla_baseline(max_seq_len=64) if baseline else ModelArgs(max_seq_len=64))
        x = torch.zeros(2, 1, m.d_model)
        with torch.no_grad():
            for weights in (torch.float32, torch.bfloat16):
                m = m.to(weights)
                amp[0] = True
                for capturing[0] in (False, True):
                    assert m._rows_path(x) == (weights == torch.bfloat16 or (baseline and not capturing[0]))
            amp[0] = False
            assert m._rows_path(x) == baseline  # no autocast, fp32 x, bf16 weights: torch's layer refuses it at the default dims


def test_weight_gradient_rows_do_not_overlap():
    # strides that torch's products take and mla_weight_grad refuses (rows that overlap or repeat, an inner stride, odd
    # strides) are copied, before the limits are asked; others are passed as they are
    from transformer_amd import kernels
    rows = kernels.weight_grad_rows
    b = torch.randn(16, 64, generator=torch.Generator().manual_seed(1)).to(torch.bfloat16)
    flat = b.view(-1)
    for t in (b[:1, :1].expand(9, 16), b[0, :16].expand(9, 16), b[:, :1].expand(16, 16), b.t(), b[:, ::2], b[:, 1:17],
              flat.as_strided((9, 16), (8, 1)), flat.as_strided((9, 16), (20, 1))):
        r = rows(t)
        assert torch.equal(r, t) and r.stride(1) == 1 and r.stride(0) >= r.size(1) and r.stride(0) % 8 == 0
    for t in (b, b[:, 8:40], b[:1, :16]):
        assert rows(t) is t


def test_contiguous_rows_off_the_alignment_are_copied():
    # a slice of a flat buffer at an odd offset is contiguous: contiguous() returns it as it is, and every entry point
    # refuses an operand that is not 16-byte aligned
    from transformer_amd import kernels
    flat = torch.arange(200, dtype=torch.float32).to(torch.bfloat16)
    for t in (flat[1:129].view(8, 16), flat[3:131].view(2, 4, 16)):
        a = kernels._aligned4(t, 8)
        assert a.data_ptr() % 16 == 0 and a.is_contiguous() and torch.equal(a, t)
    assert kernels.weight_grad_rows(flat[1:129].view(8, 16)).data_ptr() % 16 == 0
    whole = flat[8:136].view(8, 16)
    assert kernels._aligned4(whole, 8) is whole


def test_training_branch_asks_replaced_layers_nothing_but_their_call(monkeypatch):
    # a Sequential around a layer has neither in_features nor a weight
    from transformer_amd import MLA, ModelArgs, training
    monkeypatch.setattr(training, "plain_call", lambda *t: True)  # (CPU tensors)
    for name in ("q_up", "k_up", "v_up"):
        m = MLA(ModelArgs(d_model=256, n_heads=2, d_latent=128, q_lora_rank=128, max_seq_len=64)).to(torch.bfloat16)
        d = torch.zeros(1, 4, 128 + 4 * 64 + 128, dtype=torch.bfloat16)
        assert training.takes_attention(m, d)
        m._modules[name] = torch.nn.Sequential(m._modules[name])
        assert not training.takes_attention(m, d)
        assert not training.takes(m._modules[name], d[..., :128])


@pytest.mark.parametrize("n_outputs", [1, 3])
def test_undefined_gradients_reach_the_formulas_as_zeros(monkeypatch, n_outputs):
    # a consumer whose backward returns None leaves the gradient undefined: the registered operators' autograd makes zeros
    # of it, and so does the autograd.Function in their place (of the first output alone: the others have no gradient)
    from transformer_amd import kernels
    seen = []

    def body(x):
        y = x * 2
        return y if n_outputs == 1 else (y, x.sum(), x.amax())

    def setup(ctx, inputs, output):
        if n_outputs > 1:
            ctx.mark_non_differentiable(*output[1:])

    def backward(ctx, grad, *others):
        assert not kernels.batched_grad(grad)
        seen.append((grad.clone(), others))
        return grad * 2

    monkeypatch.setitem(kernels._BODIES, "probe", body)
    monkeypatch.setitem(kernels._FORMULAS, "probe", (setup, backward))
    fn = kernels._function("probe")

    class NoGrad(torch.autograd.Function):
        @staticmethod
        def forward(ctx, x):
            return x + 1

        @staticmethod
        def backward(ctx, g):
            return None

    for wrap, want in ((NoGrad.apply, 0.0), (lambda t: t + 1, 1.0)):
        x = torch.ones(2, 3, requires_grad=True)
        y = fn.apply(x)
        wrap(y if n_outputs == 1 else y[0]).sum().backward()
        grad, others = seen.pop()
        assert torch.equal(grad, torch.full((2, 3), want)) and all(o is None for o in others)
        assert torch.equal(x.grad, 2 * grad)


def test_autocast_does_not_cast_float64_inputs(monkeypatch):
    # torch's layers refuse a float64 (or integer) input beside autocast's bf16 weight, and the training branch leaves it to them
    from transformer_amd import MLA, ModelArgs, training
    monkeypatch.setattr(torch, "is_autocast_enabled", lambda *a: True)  # (no GPU: torch turns autocast off)
    monkeypatch.setattr(torch, "get_autocast_dtype", lambda *a: torch.bfloat16)
    monkeypatch.setattr(training, "plain_call", lambda *t: True)
    taken = []
    monkeypatch.setattr(training, "linear", lambda x, *ws, **k: taken.append(x.dtype))
    m = MLA(ModelArgs(d_model=256, n_heads=2, d_latent=128, q_lora_rank=128, max_seq_len=64))
    for dt in (torch.bfloat16, torch.float32, torch.float64, torch.int32):
        x = torch.zeros(2, 3, 256, dtype=dt)
        ok = dt in (torch.bfloat16, torch.float32)
        assert training.takes(m.o_proj, x) == ok
        if ok:
            m._down_all(x)
        else:
            with pytest.raises(RuntimeError):
                m._down_all(x)
    assert taken == [torch.bfloat16] * 2


@pytest.mark.parametrize("name", ["q_down", "kv_down", "k_up"])
def test_weights_made_on_each_access_are_not_kept(monkeypatch, name):
    # a parametrized weight is a fresh tensor: here one at the same address with the same version counter every time, as the
    # allocator may give it, holding other values
    from transformer_amd import MLA, ModelArgs
    import torch.nn as nn
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)  # (asks a GPU)
    m = MLA(ModelArgs(d_model=256, n_heads=2, d_latent=128, q_lora_rank=128, max_seq_len=64))
    array = m._modules[name].weight.detach().numpy().copy()

    class Made(nn.Module):
        weight = property(lambda self: torch.from_numpy(array))

    x = torch.randn(2, 3, 256, generator=torch.Generator().manual_seed(1))
    with torch.no_grad():
        with monkeypatch.context() as amp:  # (no GPU: torch turns autocast off)
            amp.setattr(torch, "is_autocast_enabled", lambda *a: True)
            amp.setattr(torch, "get_autocast_dtype", lambda *a: torch.bfloat16)
            assert m._auto_graph_ok(x[:, :1])
            m._modules[name] = Made()
            assert not m._auto_graph_ok(x[:, :1])
        for scale in (1, 2, 4):
            array *= scale
            kept = m._cached_weight("down" if name != "k_up" else "k_up:t", lambda: m._modules[name].weight, torch.float64)
            assert torch.equal(kept, torch.from_numpy(array).double())
            if name != "k_up":
                want = torch.cat([m._modules[n].weight for n in ("q_down", "qk_rope", "kv_down")], 0)
                torch.testing.assert_close(m._down_all(x), x @ want.t())
