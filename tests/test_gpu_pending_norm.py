"""Steps of one token whose products make their own norms, against the same steps with the norms as launches of their own: the same bits, call by call, from
launch lists and from graphs, over layers that exchange the stream's two rows."""
import numpy as np
import pytest

from gpu_util import make_runner

pytestmark = pytest.mark.gpu


def folder(path, hidden, inter, layers):
    from zse_amd.weights import write_random_model
    cfg = dict(architectures=["Gemma2ForCausalLM"], model_type="gemma2", num_hidden_layers=layers, hidden_size=hidden, num_attention_heads=8,
               num_key_value_heads=2, head_dim=64, query_pre_attn_scalar=64, intermediate_size=inter, vocab_size=512, rope_theta=10000.0,
               sliding_window=8, attn_logit_softcapping=50.0, final_logit_softcapping=30.0, rms_norm_eps=1e-6, max_position_embeddings=512)
    write_random_model(str(path), cfg, seed=hidden, std=0.7 * hidden ** -0.5, gain_std=0.2, dtype="bfloat16", std_of={"embed_tokens": 0.02})
    return str(path)


def decoded(runner):
    """Logits of two requests' tokens, one at a time: every step has one row."""
    from zse_amd.engine.runner import StepEntry
    rng, rows = np.random.default_rng(3), []
    for req, n in (("a", 11), ("b", 1)):
        rows.append(runner.step([StepEntry(req, rng.integers(0, 512, n).tolist(), [n - 1])]).copy())
    for i in range(8):
        rows.append(runner.step([StepEntry("ab"[i % 2], [int(rng.integers(0, 512))], [0])]).copy())
    return np.concatenate(rows)


# rows by the narrow norm's order of sums and the wide one's; down products in ranges of K, whose sums wait for the next layer
@pytest.mark.parametrize("hidden,inter,layers", [(512, 4096, 3), (1280, 4096, 2), (2048, 8192, 3)])
def test_same_bits(hidden, inter, layers, tmp_path, monkeypatch):
    from zse_amd.parts.ops import PendingNorm
    model, made = folder(tmp_path, hidden, inter, layers), []
    init, possible = PendingNorm.__init__, PendingNorm.possible
    monkeypatch.setattr(PendingNorm, "__init__", lambda self, ctx, sub, *a: (made.append(sub.layout), init(self, ctx, sub, *a))[1])
    modes = dict(calls=dict(use_graphs=False, use_steplists=False), lists=dict(use_graphs=False, use_steplists=True), graphs=dict(use_graphs=True))
    got = {}
    for waits in (True, False):
        monkeypatch.setattr(PendingNorm, "possible", staticmethod(possible if waits else lambda *a: False))
        for name, kw in modes.items():
            made.clear()
            runner = make_runner(model, "bfloat16", cache_tokens=256, max_seqs=4, max_batch_tokens=64, max_model_len=128, **kw)
            got[name, waits] = decoded(runner)
            assert (runner.steplist_runs > 0) == (name == "lists") or name == "graphs"
            assert (runner.graph_runs > 0) == (name == "graphs")
            # one a layer in front of the gated product, one between two layers
            assert set(made) == ({"rows", "parts"} if waits else set())
            if name == "calls" and waits:
                assert len(made) % (2 * layers - 1) == 0
    first = got["calls", False]
    assert np.isfinite(first).all() and np.ptp(first) > 1e-3
    for key, z in got.items():
        assert np.array_equal(z, first), key


def test_a_routed_layers_plane(tmp_path, monkeypatch):
    """A routed layer's float plane lies in the step's own memory, and behind it a layer whose q | k | v row is wider than all of that layer's buffers."""
    from zse_amd.config import (Architecture, AttentionSpec, BlockSpec, EmbeddingSpec, GatedMLPSpec, HeadSpec, LayerCall, ModelPlan, NormSpec, RotarySpec,
                                register_architecture, unregister_architecture)
    from zse_amd.config.plan import RoutedMLPSpec
    from zse_amd.engine.loading import load_model
    from zse_amd.engine.runner import StepRunner
    from zse_amd.parts.ops import PendingNorm
    from zse_amd.runtime.device import Runtime
    from zse_amd.weights import write_random_model
    H, V = 512, 512

    def block(l, ffn, nh, nkv, hd):
        norms = {r: NormSpec(H, 1e-6, True, f"l{l}.{r}") for r in ("pre_mixer", "post_mixer", "pre_ffn", "post_ffn")}
        mixer = AttentionSpec(H, nh, nkv, hd, hd ** -0.5, None, None, RotarySpec(hd, hd, 1000.0), {r: f"l{l}.attn.{r}" for r in "qkvo"})
        return BlockSpec("sandwich", mixer, ffn, norms)

    def plan_of(cfg):
        routed = RoutedMLPSpec(H, 32, 4, 2, "silu", None, "l0.router", "l0.e{e}.{role}", scale_input=False)
        gated = GatedMLPSpec(H, 1024, "silu", {r: f"l1.{r}" for r in ("gate", "up", "down")})
        return ModelPlan("PlaneLM", H, V, 256, EmbeddingSpec(V, H, 1.0, "emb"), (block(0, routed, 2, 1, 16), block(1, gated, 32, 16, 64)),
                         (LayerCall(0), LayerCall(1)), NormSpec(H, 1e-6, True, "final"), HeadSpec(V, H, None, "emb"))

    register_architecture(Architecture("PlaneLM", lambda cfg: cfg, plan_of))
    try:
        path = str(tmp_path)
        write_random_model(path, dict(architectures=["PlaneLM"]), seed=4, std=0.04, gain_std=0.1, dtype="bfloat16", std_of={"emb": 0.02})
        rt, got, possible = Runtime.get(), [], PendingNorm.possible
        for waits in (True, False):
            monkeypatch.setattr(PendingNorm, "possible", staticmethod(possible if waits else lambda *a: False))
            runner = StepRunner(load_model(path, "bfloat16", rt), rt, "bfloat16", cache_tokens=256, max_seqs=4, max_batch_tokens=64, use_graphs=False)
            got.append(decoded(runner))
        assert np.isfinite(got[0]).all() and np.array_equal(*got)
    finally:
        unregister_architecture("PlaneLM")
