"""Prompt layers whose o / down sums are added up together with the residual and the norm."""
import pytest
import torch

from copilot_for_consensus_amd.models.decoder import DecoderModel, DecoderWeights, get_config
from copilot_for_consensus_amd.ops import kernels as K
from copilot_for_consensus_amd.runtime.engine import LLMEngine
from copilot_for_consensus_amd.runtime.kv_cache import PagedKVCache


@pytest.mark.gpu
@pytest.mark.parametrize("lens", [(3,), (24,), (100, 28), (129,), (150, 131, 60), (400,)])
def test_same_logits_as_with_separate_launches(lens, monkeypatch):
    """Bit for bit: the slabs are added in the same order, the sum is rounded, added to the residual and rounded again.
    Rows of the decode GEMM (up to 128) and of the one for a few hundred rows."""
    monkeypatch.setattr(K, "prompt_plan", lambda M, N, Kd, kind="act": (0, 128, 2) if M > 128 else None)
    w = DecoderWeights.random(get_config("tiny"), "cuda", seed=5)
    m = DecoderModel(w)
    g = torch.Generator().manual_seed(sum(lens))
    prompts = [[1] + torch.randint(3, w.cfg.vocab_size, (n - 1,), generator=g).tolist() for n in lens]

    def logits():
        kv = PagedKVCache(w.cfg.layers, 64, w.cfg.kv_heads, w.cfg.head_dim, "cuda")
        eng = LLMEngine(m, kv, max_prefill_tokens=512, use_graph=False)
        seen, real = [], m.logits
        m.logits = lambda h: seen.append(real(h)) or seen[-1]
        try:
            eng.generate(prompts, max_new_tokens=1, ignore_eos=True)
        finally:
            m.logits = real
        return seen[0].clone()
    used, real = [], m._slabs_norm
    m._slabs_norm = lambda *a: used.append(real(*a)) or used[-1]
    got = logits()
    took = sum(h is not None for h in used)
    m._slabs_norm = lambda *a: None
    assert torch.equal(got, logits())
    assert took == 2 * w.cfg.layers - 1      # all but the last layer's down, whose norm reads a few rows only
