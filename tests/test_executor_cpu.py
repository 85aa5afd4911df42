"""GPT pattern lowering (CPU): which layer lists the fused executor accepts."""
import copy

import pytest

import bench
from penroz.models.executor import GPTExecutor
from penroz.models.mapper import Mapper
from penroz.models.model import NeuralNetworkModel


def _model(layers):
    return NeuralNetworkModel("x", Mapper(layers, {"adamw": {"lr": 1e-3}}))


def test_reference_example_layout_matches():
    spec = GPTExecutor.match(_model(bench.gpt2_layers(V=128, C=128, L=2, H=2, P=64)))
    assert spec is not None and (spec.C, spec.H, spec.D, spec.F, spec.V, spec.P) == (128, 2, 64, 512, 128, 64)
    assert len(spec.blocks) == 2 and spec.gelu_approx == "none"


def test_hf_style_layouts():
    from transformers import GPT2Config
    from penroz.models import hf
    cfg = GPT2Config(vocab_size=128, n_positions=64, n_embd=128, n_layer=1, n_head=2)
    spec = GPTExecutor.match(_model(hf.gpt2_layers(cfg)))  # HF default dropout 0.1: fused kernels
    assert spec is not None and spec.p_embd == 0.1 and spec.blocks[0].p_attn_res == spec.blocks[0].p_mlp_res == 0.1
    bf = _model(hf.gpt2_layers(cfg)).to(dtype=__import__("torch").bfloat16)  # /import/ loads bf16 weights
    assert GPTExecutor.match(bf).param_dtype == __import__("torch").bfloat16
    assert GPTExecutor.match(bf, require_fp32=True) is None
    cfg = GPT2Config(vocab_size=128, n_positions=64, n_embd=128, n_layer=1, n_head=2, resid_pdrop=0.0,
                     embd_pdrop=0.0, attn_pdrop=0.1)
    spec = GPTExecutor.match(_model(hf.gpt2_layers(cfg)))
    assert spec is not None and spec.gelu_approx == "tanh"  # attention dropout runs in the flash kernel


def test_non_matching_layouts():
    base = bench.gpt2_layers(V=128, C=128, L=1, H=2, P=64)
    rope = copy.deepcopy(base)
    rope[2]["residual"][0]["sequential"][2]["attention"]["rope_theta"] = 10000.0
    assert GPTExecutor.match(_model(rope)) is None
    odd_head = copy.deepcopy(base)
    odd_head[2]["residual"][0]["sequential"][2]["attention"]["num_heads"] = 4  # D = 32
    assert GPTExecutor.match(_model(odd_head)) is None
    mlp = [{"linear": {"in_features": 4, "out_features": 4}}, {"relu": {}}, {"linear": {"in_features": 4, "out_features": 2}}]
    assert GPTExecutor.match(_model(mlp)) is None


def test_head_chunk_policy(monkeypatch):
    from penroz.models.executor import _head_chunk_rows
    monkeypatch.delenv("PENROZ_HEAD_CHUNK", raising=False)
    assert _head_chunk_rows(65536, 50304) == 65536          # 6.6 GB of logits: one chunk
    c = _head_chunk_rows(4 * 65536, 50304)                   # 26 GB: ~2 GiB chunks
    assert c % 1024 == 0 and 1024 <= c < 4 * 65536 and c * 50304 * 2 <= 2 * 2**30
    monkeypatch.setenv("PENROZ_HEAD_CHUNK", "8192")
    assert _head_chunk_rows(65536, 50304) == 8192
    monkeypatch.setenv("PENROZ_HEAD_CHUNK", "0")
    assert _head_chunk_rows(4 * 65536, 50304) == 4 * 65536


def test_gemma_executor_pattern_match_modes():
    """The fused Gemma executor's pattern match (CPU): Gemma 3 / 2 / 1 layer lists map to the
    combine modes 0 / 1 / 2; a tied head or a GPT layer list does not match."""
    from types import SimpleNamespace
    from penroz.models.gemma_executor import GemmaExecutor
    from penroz.models.mapper import Mapper
    from penroz.models.model import NeuralNetworkModel
    for mt, mode in (("gemma3_text", 0), ("gemma2", 1), ("gemma", 2)):
        cfg = SimpleNamespace(model_type=mt, vocab_size=64, hidden_size=64, intermediate_size=128, num_hidden_layers=2,
                              num_attention_heads=2, num_key_value_heads=1, head_dim=64, rms_norm_eps=1e-6,
                              rope_theta=10000.0, attention_dropout=0.0, hidden_activation="gelu_pytorch_tanh")
        m = NeuralNetworkModel("g", Mapper(Mapper.from_hf_config(cfg), {"adamw": {"lr": 1e-3}}))
        spec = GemmaExecutor.match(m)
        assert spec is not None and spec.mode == mode and spec.F == 128 and spec.act == 1
        m.layers[-2].weight = m.layers[0].weight  # tied head: not lowered
        assert GemmaExecutor.match(m) is None
    import bench
    g = NeuralNetworkModel("t", Mapper(bench.gpt2_layers(V=64, C=64, L=1, H=1, P=32), {"adamw": {"lr": 1e-3}}))
    assert GemmaExecutor.match(g) is None


def test_gemma_executor_matches_heterogeneous_gemma4_layer_list():
    """Gemma 4 layer lists (reference mappers.py:206-233) lower to the fused executor with
    per-block shapes: global_head_dim / KV heads on full-attention layers, double-wide MLPs on
    KV-shared layers; C up to 6144 (Gemma-3 27B: 5376)."""
    from types import SimpleNamespace
    from penroz.models.gemma_executor import GemmaExecutor
    from penroz.models.mapper import Mapper
    from penroz.models.model import NeuralNetworkModel
    cfg = SimpleNamespace(model_type="gemma4", vocab_size=64, hidden_size=64, intermediate_size=128,
                          num_hidden_layers=4, num_attention_heads=2, num_key_value_heads=2, head_dim=64,
                          rms_norm_eps=1e-6, rope_theta=10000.0, attention_dropout=0.0,
                          hidden_activation="gelu_pytorch_tanh",
                          layer_types=["sliding_attention", "full_attention"] * 2, global_head_dim=128,
                          num_global_key_value_heads=1, num_kv_shared_layers=2, use_double_wide_mlp=True)
    m = NeuralNetworkModel("g4", Mapper(Mapper.from_hf_config(cfg), {"adamw": {"lr": 1e-3}}))
    spec = GemmaExecutor.match(m)
    assert spec is not None and not spec.uniform
    assert [(b.H, b.Hkv, b.D, b.F) for b in spec.blocks] == [(2, 2, 64, 128), (2, 1, 128, 128), (2, 2, 64, 256),
                                                            (2, 1, 128, 256)]
    wide = SimpleNamespace(**{**vars(cfg), "hidden_size": 5376, "num_hidden_layers": 1, "layer_types": None,
                              "intermediate_size": 64, "vocab_size": 16})
    assert GemmaExecutor.match(NeuralNetworkModel("w", Mapper(Mapper.from_hf_config(wide), {"adamw": {}}))) is not None


def _range_exec(monkeypatch):
    """A bare executor with only the weight-gradient bookkeeping live: flat fp32 buffer, wgrad
    done eagerly on the CPU (g = dyᵀ·x or g += dyᵀ·x), no side stream."""
    import types
    import torch
    from penroz.models import executor as E
    ex = object.__new__(GPTExecutor)
    ex.flat_grad = torch.zeros(64)
    ex.device = types.SimpleNamespace(type="cuda", index=0)  # range learning is a GPU-path feature
    ex._side = None
    ex.wait_gradients = lambda: None

    def wgrad(dy, x, g, acc):
        r = dy.t() @ x
        if acc:
            g.add_(r)
        else:
            g.copy_(r)
    monkeypatch.setattr(E.gemm_ops, "wgrad", wgrad)
    return ex


def test_wgrad_ranges_chunked_after_learning(monkeypatch):
    """After the ranges are learned, a key that writes sub-ranges (chunked wgrad) must
    never accumulate onto last step's data — whether its first chunk is a sub-range, the whole
    learned range, or some parts are never written."""
    import torch
    ex = _range_exec(monkeypatch)
    torch.manual_seed(0)
    A = ex.flat_grad[0:32].view(8, 4)    # weight A's gradient
    Bg = ex.flat_grad[40:56].view(4, 4)  # weight B's gradient; [32:40) and [56:64) are other grads
    dyA, xA = torch.randn(5, 8), torch.randn(5, 4)
    dyB, xB = torch.randn(5, 4), torch.randn(5, 4)
    # learning step: whole-range writes
    ex.zero_grad()
    ex._wgrad_into(1, dyA, xA, A)
    ex._wgrad_into(2, dyB, xB, Bg)
    ex._finish_wgrad_bookkeeping()
    assert ex._zero_gaps == [(0 + 32, 40), (56, 64)]
    assert torch.allclose(A, dyA.t() @ xA)

    def step(writes_a, learned_ranges_skipped=False):
        ex.flat_grad.fill_(123.0)  # last step's values everywhere
        ex.zero_grad()
        assert torch.all(ex.flat_grad[32:40] == 0)
        if learned_ranges_skipped:
            assert torch.all(ex.flat_grad[40:56] == 123.0) and torch.all(ex.flat_grad[0:32] == 123.0)
        for r0, r1, dy, x in writes_a:
            ex._wgrad_into(1, dy[:, r0:r1], x, A[r0:r1])
        ex._wgrad_into(2, dyB, xB, Bg)
        ex._finish_wgrad_bookkeeping()
        assert torch.allclose(Bg, dyB.t() @ xB)

    d1, d2 = torch.randn(5, 8), torch.randn(5, 8)
    # sub-ranges first, one range accumulated twice (two token chunks), the rest once
    step([(0, 4, d1, xA), (0, 4, d2, xA), (4, 8, d1, xA)], learned_ranges_skipped=True)
    want = torch.cat([(d1[:, :4] + d2[:, :4]).t() @ xA, d1[:, 4:].t() @ xA])
    assert torch.allclose(A, want, atol=1e-5)
    # the whole learned range first (overwrite), then a sub-range accumulates onto it; with the
    # pattern changed zero_grad now clears everything, so re-arm the skip to test the stale path
    assert ex._zero_gaps is None
    ex._zero_gaps = [(32, 40), (56, 64)]
    step([(0, 8, d1, xA), (2, 6, d2, xA)], learned_ranges_skipped=True)
    want = d1.t() @ xA
    want[2:6] += d2[:, 2:6].t() @ xA
    assert torch.allclose(A, want, atol=1e-5)
    # a part never written this step ends up zero, not stale
    ex._zero_gaps = [(32, 40), (56, 64)]
    step([(0, 3, d1, xA)], learned_ranges_skipped=True)
    assert torch.allclose(A[0:3], d1[:, :3].t() @ xA, atol=1e-5) and torch.all(A[3:] == 0)
    # the changed pattern makes zero_grad clear everything from now on
    assert ex._wgrad_ranges_invalid and ex._zero_gaps is None


def test_side_stream_cu_mask_words():
    from penroz.models.executor import cu_mask_words
    w = cu_mask_words("stride:4", 256)
    assert len(w) == 8 and all(x == 0x11111111 for x in w)
    w = cu_mask_words("stride:8:1", 256)
    assert all(x == 0x02020202 for x in w)
    assert cu_mask_words("first:40", 256)[:2] == [0xFFFFFFFF, 0xFF] and cu_mask_words("first:40", 256)[2:] == [0] * 6
    with pytest.raises(ValueError):
        cu_mask_words("half", 256)


def test_zero_gap_minus_skip_range():
    from penroz.models.executor import _minus
    assert _minus([(0, 10), (20, 30)], None) == [(0, 10), (20, 30)]
    assert _minus([(0, 10), (20, 30)], (5, 25)) == [(0, 5), (25, 30)]
    assert _minus([(0, 10)], (0, 10)) == []
    assert _minus([(0, 100)], (40, 60)) == [(0, 40), (60, 100)]
    assert _minus([(10, 20)], (30, 40)) == [(10, 20)]


class _Stream:
    """A stream that notes what waits for what."""

    def __init__(self, cuda_stream, log):
        self.cuda_stream, self.log = cuda_stream, log

    def wait_stream(self, other):
        self.log.append((self.cuda_stream, other.cuda_stream))


def test_a_failed_step_defers_nothing_to_the_next(monkeypatch):
    """A step on two streams that raises in its backward, then one on a single stream: the second step's reductions stay
    on the main stream, which has waited for the side stream."""
    from types import SimpleNamespace

    import torch
    from penroz.models import executor
    waits, deferred = [], []
    main = _Stream(1, waits)
    monkeypatch.setattr(executor._ext, "kernels", lambda: SimpleNamespace(
        set_deferred_reduce_stream=lambda stream, device: deferred.append(stream)))
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: main)
    ex = GPTExecutor.__new__(GPTExecutor)
    ex.device, ex.flat, ex._opt_flat, ex.reducer = torch.device("cuda", 0), torch.empty(10), False, None
    ex._side_stream, ex._buf_free, seen = _Stream(7, waits), {1: "event"}, []

    def micro(idx, targets, scale, sync, capture):
        ex._plan_step(idx.numel())
        ex._defer_reductions(True)
        seen.append(deferred[-1] if deferred else 0)
        if ex._side is not None:
            raise MemoryError("in the backward")
        ex._defer_reductions(False)
        ex._join_side()

    ex._train_micro_step = micro
    ex.SIDE_MIN_FLOPS = 6 * 100 * 10
    with pytest.raises(MemoryError):
        ex.train_micro_step(torch.empty(4, 64), None, 1.0)
    assert deferred[-1] == 0 and waits == [(1, 7)] and not ex._buf_free
    deferred.append(7)  # whatever was left of it
    ex.train_micro_step(torch.empty(1, 64), None, 1.0)
    assert seen == [7, 0] and deferred[-1] == 0


def test_deferred_reductions_are_a_threads_own():
    """One thread's executor defers its reductions, another's does not."""
    import threading

    from penroz.ops import _ext
    if not _ext.available("penroz_kernels"):
        pytest.skip("extension not built")
    k, seen = _ext.kernels(), []
    k.set_deferred_reduce_stream(64, 0)
    try:
        t = threading.Thread(target=lambda: seen.append(k.get_deferred_reduce_stream()))
        t.start()
        t.join()
        assert seen == [0] and k.get_deferred_reduce_stream() == 64
    finally:
        k.set_deferred_reduce_stream(0, 0)


# layers, parameters, tokens, ms per step on two streams / on one
SIDE_STREAM_MS = [
    (12, 163109376, 256, 9.0, 5.2), (12, 163109376, 2048, 9.3, 7.2), (12, 163109376, 4096, 9.7, 9.4),
    (12, 163109376, 6144, 11.1, 11.7), (12, 163109376, 65536, 62.0, 63.7), (4, 106406400, 1024, 3.4, 2.7),
    (4, 106406400, 3072, 3.8, 4.0), (24, 406382592, 2048, 18.1, 15.9), (24, 406382592, 5120, 24.0, 24.3),
    (48, 1638172800, 512, 34.7, 32.1), (48, 1638172800, 1024, 36.2, 39.0), (6, 17332224, 8192, 4.9, 3.6),
    (26, 1301862528, 256, 20.6, 19.4), (26, 1301862528, 512, 20.9, 22.2), (18, 435861120, 1024, 14.5, 12.4),
    (18, 435861120, 3072, 15.8, 17.3), (8, 818713728, 64, 7.8, 8.1)]


@pytest.mark.parametrize("layers,params,tokens,two,one", SIDE_STREAM_MS)
def test_steps_take_the_streams_measured_faster(layers, params, tokens, two, one):
    import torch
    ex = GPTExecutor.__new__(GPTExecutor)
    ex.L, ex._side_stream = layers, "side"
    ex.flat = torch.empty(params, device="meta")
    ex._plan_step(tokens)
    assert (ex._side is not None) == (two < one)


def test_the_stream_rule_counts_the_models_own_parameters():
    import torch
    with torch.device("meta"):
        m = _model(bench.gpt2_layers())
    assert sum(p.numel() for p in m.parameters()) == SIDE_STREAM_MS[0][1]


@pytest.mark.parametrize("gathered", [False, True])
@pytest.mark.parametrize("two", [False, True])
def test_weight_gradients_beside_a_second_stream_are_planned_so(monkeypatch, gathered, two):
    """The rule of the weight gradients' kernel is told of the main stream's work, whether a layer's products are gathered
    or go out one by one."""
    import contextlib
    from types import SimpleNamespace

    import torch
    from penroz.models import executor as E
    from penroz.ops import gemm
    seen = []
    monkeypatch.setattr(gemm, "_native_wgrad", lambda dy, x: True)
    monkeypatch.setattr(gemm, "kernels", lambda: SimpleNamespace(
        wgrad_group=lambda dys, xs, grads, accumulate, variant, shared=False: seen.append((len(dys), shared))))
    event = SimpleNamespace(record=lambda stream: None)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: None)
    monkeypatch.setattr(torch.cuda, "Event", lambda: event)
    monkeypatch.setattr(torch.cuda, "stream", lambda stream: contextlib.nullcontext())
    ex = object.__new__(E.GPTExecutor)
    ex.device, ex._buf_free = None, {}
    ex._side = SimpleNamespace(wait_event=lambda e: None) if two else None
    ex._wgrad_queue = [] if gathered else None
    for _ in range(2):
        ex._emit_wgrad(torch.empty(4, 8), torch.empty(4, 8), torch.empty(8, 8), True)
    ex._flush_wgrads()
    assert seen == ([(2, two)] if gathered else [(1, two)] * 2)


@pytest.mark.parametrize("tokens,two,one", [(256, 16.3, 16.0), (512, 18.5, 18.6), (1024, 22.4, 23.6), (1536, 27.0, 28.3),
                                            (2048, 28.6, 30.1), (4096, 42.5, 44.0), (8192, 66.4, 69.1)])
def test_gemma_steps_take_the_streams_measured_faster(tokens, two, one):
    import torch
    from penroz.models.gemma_executor import GemmaExecutor
    ex = GemmaExecutor.__new__(GemmaExecutor)  # Gemma-3 1B
    ex.L, ex._side_stream, ex.flat = 26, "side", torch.empty(1301862528, device="meta")
    ex._plan_step(tokens)
    assert (ex._side is not None) == (two < one)


def test_gemma_products_that_no_launch_takes_together_start_at_once(monkeypatch):
    """On two streams, in steps of up to 4096 tokens; one stream, larger steps and products of one launch: gathered."""
    from penroz.models import executor as E
    from penroz.models.gemma_executor import GemmaExecutor
    shapes = ((8, 8), (16, 8))
    monkeypatch.setattr(E.gemm_ops, "wgrad_together", lambda sh, tokens, device, shared: (sh, shared) == ("one", True))
    ex = GemmaExecutor.__new__(GemmaExecutor)
    ex.device, ex._shapes_by_layer = None, [shapes, "one"]
    for side, l, tokens, gathered in [("side", 0, 2048, False), ("side", 1, 2048, True), (None, 0, 2048, True),
                                      ("side", 0, 4095, False), ("side", 0, 4096, True), (None, 0, 16384, True),
                                      (None, 0, 16385, False)]:
        ex._side = side
        ex._gather_wgrads(l, tokens)
        assert (ex._wgrad_queue is not None) == gathered


def test_gemma_layer_shapes_are_those_of_its_weight_gradients():
    from types import SimpleNamespace

    from penroz.models.gemma_executor import GemmaExecutor
    cfg = SimpleNamespace(model_type="gemma3_text", vocab_size=64, hidden_size=64, intermediate_size=128, num_hidden_layers=1,
                          num_attention_heads=2, num_key_value_heads=1, head_dim=64, rms_norm_eps=1e-6,
                          rope_theta=10000.0, attention_dropout=0.0, hidden_activation="gelu_pytorch_tanh")
    spec = GemmaExecutor.match(NeuralNetworkModel("g", Mapper(Mapper.from_hf_config(cfg), {"adamw": {"lr": 1e-3}})))
    assert GemmaExecutor._wgrad_shapes(spec.blocks[0]) == ((64, 128), (64, 128), (256, 64), (256, 64))
    gpt = GPTExecutor.match(_model(bench.gpt2_layers(V=128, C=128, L=1, H=2, P=64)))
    assert GPTExecutor._wgrad_shapes(gpt.blocks[0]) == ((128, 512), (512, 128), (128, 128), (384, 128))
