"""The products around a chunk over a cache, at sizes off the tiles."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("weights", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("dims", ["baseline", "default"])
@pytest.mark.parametrize("B,T,L", [(1, 2, 5), (3, 13, 70), (2, 129, 33), (2, 33, 0)])
def test_chunk_equals_the_same_layer_with_hooks(B, T, L, dims, weights):
    """A hook on k_up keeps it a product of its own; the absorbed form has none to keep, so it is also compared with the
    form over per-head K and V.  bf16 operands, stored K, V and outputs: a few roundings of 2^-9 each way."""
    from contextlib import nullcontext
    from transformer_amd import MLA, ModelArgs, mla
    torch.manual_seed(3)
    with torch.device("cuda"):
        m = MLA(ModelArgs.mla_baseline() if dims == "baseline" else ModelArgs())  # bf16 RoPE tables
        m = m.to(weights) if weights == torch.bfloat16 else m
        x = torch.randn(B, T, m.d_model).to(weights)
        cache = None
        if L:
            cache = {"latent": torch.randn(B, L, m.d_latent).bfloat16(),
                     "k_rope": torch.randn(B, m.n_k_rope_heads, L, 64).bfloat16(), "seq_len": L}
    amp = nullcontext() if weights == torch.bfloat16 else torch.autocast("cuda", torch.bfloat16)
    with torch.no_grad(), amp:
        y = m(x, cache, True)[0]
        h = m.k_up.register_forward_hook(lambda *a: None)
        old, mla.ABSORBED_PREFILL = mla.ABSORBED_PREFILL, False
        try:
            want = m(x, cache, True)[0]
        finally:
            mla.ABSORBED_PREFILL = old
            h.remove()
        assert y.shape == want.shape and y.dtype == want.dtype
        assert (y.double() - want.double()).norm() <= 8 * 2.0 ** -9 * want.double().norm()
        m.v_up.weight.mul_(2)  # the kept weights follow
        assert not torch.equal(m(x, cache, True)[0], y)


def test_recorded_chunk_follows_its_weights():
    """A recorded chunk reads k_up and v_up themselves: replays after an update give the updated layer's outputs."""
    from transformer_amd import MLA, ModelArgs
    torch.manual_seed(4)
    with torch.device("cuda"):
        m = MLA(ModelArgs()).to(torch.bfloat16)
        x = torch.randn(1, 9, m.d_model).bfloat16()
        cache = {"latent": torch.randn(1, 40, m.d_latent).bfloat16(),
                 "k_rope": torch.randn(1, m.n_k_rope_heads, 40, 64).bfloat16(), "seq_len": 40}
    with torch.no_grad():
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            for _ in range(2):
                m(x, dict(cache), True)
        torch.cuda.current_stream().wait_stream(s)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y = m(x, dict(cache), True)[0]
        for _ in range(3):
            graph.replay()
            want = m(x, dict(cache), True)[0]
            assert (y.double() - want.double()).norm() <= 4 * 2.0 ** -9 * want.double().norm()
            m.v_up.weight.mul_(0.5)


@pytest.mark.parametrize("dims", ["baseline", "default"])
def test_recorded_few_row_chunk_follows_fp32_projections(dims):
    """fp32 weights under autocast, at most 64 rows: replays after an update of q_up, o_proj (and, where they are layers,
    k_up and v_up) give the updated layer's outputs.  Both round bf16 weights and results: a few times 2^-9."""
    from transformer_amd import MLA, ModelArgs
    torch.manual_seed(6)
    with torch.device("cuda"):
        m = MLA(ModelArgs.mla_baseline() if dims == "baseline" else ModelArgs())
        x = torch.randn(2, 9, m.d_model)
        cache = {"latent": torch.randn(2, 40, m.d_latent).bfloat16(),
                 "k_rope": torch.randn(2, m.n_k_rope_heads, 40, 64).bfloat16(), "seq_len": 40}
    with torch.no_grad(), torch.autocast("cuda", torch.bfloat16, cache_enabled=False):
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            for _ in range(2):
                m(x, dict(cache), True)
        torch.cuda.current_stream().wait_stream(s)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y = m(x, dict(cache), True)[0]
        for i in range(4):
            graph.replay()
            want = m(x, dict(cache), True)[0]
            assert (y.double() - want.double()).norm() <= 4 * 2.0 ** -9 * want.double().norm(), i
            for name in ("q_up", "o_proj") + (("k_up", "v_up") if dims == "default" else ()):
                m._modules[name].weight.mul_(1.25 if i % 2 else 0.5)


@pytest.mark.parametrize("dims", ["baseline", "default"])
@pytest.mark.parametrize("B,T,L", [(1, 1, 30), (4, 10, 0), (2, 9, 40)])
def test_few_row_calls_run_hooked_projections(B, T, L, dims):
    """A hook on q_up that doubles its output does what doubling its weight does (exact in bf16), and one on o_proj runs."""
    from transformer_amd import MLA, ModelArgs
    torch.manual_seed(7)
    with torch.device("cuda"):
        m = MLA(ModelArgs.mla_baseline() if dims == "baseline" else ModelArgs()).to(torch.bfloat16)
        x = torch.randn(B, T, m.d_model).bfloat16()
        cache = None
        if L:
            cache = {"latent": torch.randn(B, L, m.d_latent).bfloat16(),
                     "k_rope": torch.randn(B, m.n_k_rope_heads, L, 64).bfloat16(), "seq_len": L}
    seen = []
    with torch.no_grad():
        hook = m.o_proj.register_forward_hook(lambda mod, a, y: seen.append(1))
        h = m.q_up.register_forward_hook(lambda mod, a, y: y * 2)
        y = m(x, cache, True)[0]
        h.remove()
        m.q_up.weight.mul_(2)
        want = m(x, cache, True)[0]
        hook.remove()
    assert len(seen) == 2 and torch.equal(y, want)


@pytest.mark.parametrize("weights", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T", [9, 75])
def test_chunk_sees_updates_past_the_version_counter(T, weights):
    """p.data writes do not count in p._version.  A chunk over per-head K and V reads q_up, k_up, v_up and o_proj
    themselves: doubling v_up so doubles the attention's output, exactly, and the layer's with it."""
    from contextlib import nullcontext
    from transformer_amd import MLA, ModelArgs
    torch.manual_seed(10)
    with torch.device("cuda"):
        m = MLA(ModelArgs())  # bf16 RoPE tables
        m = m.to(weights) if weights == torch.bfloat16 else m
        x = torch.randn(2, T, m.d_model).to(weights)
        cache = {"latent": torch.randn(2, 40, m.d_latent).bfloat16(),
                 "k_rope": torch.randn(2, m.n_k_rope_heads, 40, 64).bfloat16(), "seq_len": 40}
    amp = nullcontext() if weights == torch.bfloat16 else torch.autocast("cuda", torch.bfloat16, cache_enabled=False)
    with torch.no_grad(), amp:
        y = m(x, dict(cache), True)[0]
        for name in ("v_up", "o_proj"):
            m._modules[name].weight.data.mul_(2)
            y2 = m(x, dict(cache), True)[0]
            assert torch.equal(y2, 2 * y), name
            y = y2
        for name in ("q_up", "k_up"):  # other scores
            m._modules[name].weight.data.mul_(2)
            y2 = m(x, dict(cache), True)[0]
            assert not torch.equal(y2, y), name
            y = y2
    assert "kv_up" not in m.__dict__.get("_derived", {})


@pytest.mark.parametrize("weights", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,T,L", [(2, 20, None), (2, 100, 0), (2, 10, 40), (2, 70, 40), (2, 1, 40)])
def test_compiled_calls_are_one_graph_at_the_default_dims(B, T, L, weights):
    """No-cache, prompt, chunks on either side of 64 rows, one token; fullgraph raises at a graph break.  Compiled calls take
    the layers where eager ones may take the few-row kernels: a few roundings of 2^-9."""
    from contextlib import nullcontext
    from transformer_amd import MLA, ModelArgs
    torch.manual_seed(11)
    with torch.device("cuda"):
        m = MLA(ModelArgs())  # bf16 RoPE tables
        m = m.to(weights) if weights == torch.bfloat16 else m
        x = torch.randn(B, T, m.d_model).to(weights)
        cache = None
        if L:
            cache = {"latent": torch.randn(B, L, m.d_latent).bfloat16(),
                     "k_rope": torch.randn(B, m.n_k_rope_heads, L, 64).bfloat16(), "seq_len": L}
    amp = nullcontext() if weights == torch.bfloat16 else torch.autocast("cuda", torch.bfloat16)
    torch._dynamo.reset()
    with torch.no_grad(), amp:
        got = torch.compile(lambda t: m(t, cache, L is not None)[0], backend="eager", fullgraph=True)(x)
        want = m(x, cache, L is not None)[0]
    assert (got.double() - want.double()).norm() <= 8 * 2.0 ** -9 * want.double().norm()


def test_absorbed_chunk_compiles_as_it_runs():
    """The absorbed form's last product writes a view in eager mode and is a plain product under torch.compile: bit for bit."""
    from transformer_amd import MLA, ModelArgs
    torch.manual_seed(12)
    with torch.device("cuda"):
        m = MLA(ModelArgs.mla_baseline()).to(torch.bfloat16)
        x = torch.randn(2, 70, m.d_model).bfloat16()
        cache = {"latent": torch.randn(2, 40, m.d_latent).bfloat16(), "k_rope": torch.randn(2, 1, 40, 64).bfloat16(),
                 "seq_len": 40}
    torch._dynamo.reset()
    with torch.no_grad():
        reasons = [str(r.reason) for r in torch._dynamo.explain(lambda t: m(t, cache, True)[0])(x).break_reasons]
        assert not any("out=" in r for r in reasons), reasons
        got = torch.compile(lambda t: m(t, cache, True)[0], backend="eager")(x)
        assert torch.equal(got, m(x, cache, True)[0])
