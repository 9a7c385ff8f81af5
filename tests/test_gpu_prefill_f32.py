"""Prompts of f32-cache sessions as rows on the matrix cores (k_pf_attn_f32 and the
row GEMMs) against the CPU oracle and the token steps.

Bar 1e-4 (maximum difference over the largest value): activations, keys and values
carry at least 22 bits and every sum is f32, so a row of K <= 1536 products is
within about sqrt(K) 2^-24 = 2.3e-6 of the exact one, some ten such sums lie
between the embedding and the logits, and the largest of a few thousand logits'
errors is about four times their root mean square."""
import numpy as np
import pytest

import oracle
import uaii_amd
from uaii_amd import synth
from test_gpu_prefill import PREFILL_CFGS

pytestmark = pytest.mark.gpu

# one head per kv head and groups of 3 and 8 query heads: the attention block's
# other head and query splits
CFGS = dict(PREFILL_CFGS)
CFGS["mha_hd128"] = synth.ModelConfig(n_layers=2, dim=512, n_heads=4, n_kv_heads=4, ffn=512, vocab=900, ctx_len=512,
                                      type_default=uaii_amd.Q8_0, seed=61)
CFGS["group3"] = synth.ModelConfig(n_layers=2, dim=384, n_heads=6, n_kv_heads=2, ffn=512, vocab=900, ctx_len=512,
                                   type_default=uaii_amd.Q4_0, seed=62)
CFGS["group8_hd128"] = synth.ModelConfig(n_layers=2, dim=1024, n_heads=8, n_kv_heads=1, ffn=512, vocab=900,
                                         ctx_len=512, type_default=uaii_amd.Q4_0, seed=63)

# formats that prefill() does not take: the sums that Q5_K's minimums read beside a Q6_K
# V, F16's own activations beside the pairs of the other formats of a QKV group (whose
# waves are twice as wide) and of an FFN, both as experts (K = 768: a block's two wave
# groups take one and two units; F16: a K of no whole unit, and a shared expert)
OTHER_CFGS = {
    "q5_k": synth.ModelConfig(n_layers=2, dim=512, n_heads=8, n_kv_heads=2, ffn=1536, vocab=1500, ctx_len=512,
                              type_default=uaii_amd.Q5_K, type_attn_v=uaii_amd.Q6_K, type_ffn_down=uaii_amd.Q6_K,
                              seed=64),
    "q8_0_v_q5_k": synth.ModelConfig(n_layers=2, dim=512, n_heads=8, n_kv_heads=4, ffn=1024, vocab=1500, ctx_len=512,
                                     type_default=uaii_amd.Q8_0, type_attn_v=uaii_amd.Q5_K,
                                     type_ffn_down=uaii_amd.Q5_K, seed=65),
    "f16": synth.ModelConfig(n_layers=2, dim=512, n_heads=8, n_kv_heads=4, ffn=1024, vocab=1500, ctx_len=512,
                             type_default=uaii_amd.F16, seed=66),
    "q8_0_v_f16": synth.ModelConfig(n_layers=2, dim=512, n_heads=8, n_kv_heads=2, ffn=1024, vocab=1500, ctx_len=512,
                                    type_default=uaii_amd.Q8_0, type_attn_v=uaii_amd.F16,
                                    type_ffn_down=uaii_amd.F16, seed=67),
    "moe_q5_k": synth.ModelConfig(n_layers=2, dim=768, n_heads=12, n_kv_heads=4, ffn=768, vocab=1200, ctx_len=512,
                                  type_default=uaii_amd.Q5_K, n_experts=4, top_k=2, router_std=1.0 / 28, seed=68),
    "moe_f16": synth.ModelConfig(n_layers=2, dim=512, n_heads=8, n_kv_heads=2, ffn=320, vocab=1200, ctx_len=512,
                                 type_default=uaii_amd.F16, n_experts=4, top_k=2, router_std=1.0 / 22, shared_ffn=192,
                                 seed=69),
}
CFGS.update(OTHER_CFGS)


def maxrel(a, b):
    return float(np.abs(np.asarray(a) - b).max() / np.abs(b).max())


def generate(path, prompt, n_new, **kw):
    with uaii_amd.Session(path, profile=True, **kw) as s:
        ids = s.generate(prompt, n_new)
        return ids, s.get("logits"), "pf_attention" in s.profile_summary()


@pytest.mark.parametrize("n_prompt", [16, 33, 150])
@pytest.mark.parametrize("name", list(CFGS))
def test_f32_prompt_rows(name, n_prompt):
    cfg = CFGS[name]
    path = synth.cached_model(cfg)
    prompt = np.random.default_rng(cfg.seed + n_prompt).integers(0, cfg.vocab, n_prompt).astype(np.int64)
    print(name, n_prompt, flush=True)
    ids, logits, rows = generate(path, prompt, 4)
    assert rows, "the prompt should run as rows"
    want_ids, want = oracle.Model(path).generate(prompt, 4)
    assert np.array_equal(ids, want_ids)
    print("logits maxrel", maxrel(logits, want["logits"]), flush=True)
    assert maxrel(logits, want["logits"]) < 1e-4


@pytest.mark.parametrize("n_prompt", [33, 150])
@pytest.mark.parametrize("name", list(OTHER_CFGS))
def test_f16_prompt_rows(name, n_prompt):
    """The same over an f16 cache, whose prompts generate() alone runs as rows in these
    formats (bar 2e-3, as for the formats that prefill() takes)."""
    cfg = CFGS[name]
    path = synth.cached_model(cfg)
    prompt = np.random.default_rng(cfg.seed + n_prompt).integers(0, cfg.vocab, n_prompt).astype(np.int64)
    print(name, n_prompt, flush=True)
    with uaii_amd.Session(path, kv_f16=True) as s:
        assert not s.prefill_supported()
    ids, logits, rows = generate(path, prompt, 4, kv_f16=True)
    assert rows, "the prompt should run as rows"
    want_ids, want = oracle.Model(path).generate(prompt, 4, kv_f16=True)
    assert np.array_equal(ids, want_ids)
    assert maxrel(logits, want["logits"]) < 2e-3


@pytest.mark.parametrize("t", [uaii_amd.Q4_0, uaii_amd.Q5_K], ids=lambda t: uaii_amd.TYPE_NAMES[t])
def test_f32_prompt_of_two_chunks(t):
    """A prompt past the default chunk of 1024 tokens: a short second chunk over the
    first one's keys."""
    cfg = synth.ModelConfig(n_layers=2, dim=256, n_heads=4, n_kv_heads=2, ffn=512, vocab=900, ctx_len=1280,
                            type_default=t, seed=70)
    path = synth.cached_model(cfg)
    prompt = np.random.default_rng(8).integers(0, cfg.vocab, 1100).astype(np.int64)
    ids, logits, rows = generate(path, prompt, 4)
    assert rows
    want_ids, want = oracle.Model(path).generate(prompt, 4)
    assert np.array_equal(ids, want_ids)
    assert maxrel(logits, want["logits"]) < 1e-4


def test_f32_prompt_chunks(monkeypatch):
    """Chunks of 32 rows at p0 > 0 over the earlier chunks' keys."""
    cfg = CFGS["gqa_q4_0"]
    path = synth.cached_model(cfg)
    prompt = np.random.default_rng(5).integers(0, cfg.vocab, 150).astype(np.int64)
    monkeypatch.setenv("UAII_PREFILL", "0")
    want_ids, want, rows = generate(path, prompt, 4)
    assert not rows
    monkeypatch.delenv("UAII_PREFILL")
    monkeypatch.setenv("UAII_PREFILL_CHUNK", "32")
    ids, logits, rows = generate(path, prompt, 4)
    assert rows and np.array_equal(ids, want_ids) and maxrel(logits, want) < 1e-4


def test_f32_session_keeps_its_budget():
    """prefill() itself stays a f16-cache call, and a budget with no room for the
    rows' buffers runs the prompt in token steps as before."""
    cfg = CFGS["gqa_q4_0"]
    path = synth.cached_model(cfg)
    prompt = np.arange(40, dtype=np.int64) * 7 % cfg.vocab
    with uaii_amd.Session(path) as s:
        assert not s.prefill_supported()
        s.begin(prompt, 64)
        with pytest.raises(uaii_amd.UaiiError, match="not_implemented"):
            s.prefill(8)
    lo, hi = 1, 1 << 26  # KiB-wide bisection of the smallest budget that creates
    while hi - lo > 1024:
        mid = (lo + hi) // 2
        try:
            uaii_amd.Session(path, budget_bytes=mid).close()
            hi = mid
        except uaii_amd.UaiiError:
            lo = mid
    want_ids, want, rows = generate(path, prompt, 4)
    assert rows
    ids, logits, rows = generate(path, prompt, 4, budget_bytes=hi)
    assert not rows and np.array_equal(ids, want_ids) and maxrel(logits, want) < 1e-4
