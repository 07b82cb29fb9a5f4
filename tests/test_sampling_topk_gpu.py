"""The device sampler's top-k route at the edges of its rule: vocabularies
around its group sizes, k on both sides of nine tenths of the group count, and
logits with so many equal values that the threshold leaves more candidates
than the workgroup's list holds.

The logits are planted: every LM-head row (F32) has one nonzero weight, in one
column, so a row's logit is one f32 product.  The drawn token must be that of
the float64 restatement, ties in ascending token order; draws and cutoffs
within 1e-5 of a boundary are left out (the sums are f32 in another order).
"""
from __future__ import annotations

import numpy as np
import pytest

from gguf_write import rewrite
from hf_checkpoint import gguf_names
from test_sampling import f64_sample

pytestmark = pytest.mark.gpu


def planted(llrs, backend, tmp_path, weights):
    V = weights.size
    cfg = llrs.SynthConfig(hidden_size=64, intermediate_size=64, num_attention_heads=2, num_key_value_heads=1,
                           num_hidden_layers=1, vocab_size=V, max_position_embeddings=32,
                           recipe=llrs.LoadQuantization.NONE, seed=5, tie_word_embeddings=False)
    cfg.write_gguf(tmp_path / "src.gguf")
    head = np.zeros((V, 64), np.float32)
    head[:, 7] = weights
    rewrite(llrs, tmp_path / "src.gguf", tmp_path / "p.gguf", cfg, gguf_names(1, tied=False),
            {"output.weight": (0, V, 64, head.tobytes())})
    model = llrs.ModelLoader.load_dynamic(tmp_path / "p.gguf", backend)
    kv = llrs.KVCache(model, 16)
    model.prefill(np.array([1, 2, 3], np.uint32), 0, kv)
    return kv


def near_cutoff(logits, t, k, tp, pen, recent):
    v = np.asarray(logits, np.float64).copy()
    if pen != 1.0:
        seen = np.unique([r for r in recent if r < v.size]).astype(int)
        v[seen] = np.where(v[seen] > 0, v[seen] / pen, v[seen] * pen)
    p = np.sort(np.exp((v - v.max()) / t))[::-1][:k or None]
    return bool(np.min(np.abs(np.cumsum(p) / p.sum() - tp)) < 1e-5)


@pytest.mark.parametrize("spread", ["normal", "five_levels", "equal"])
@pytest.mark.parametrize("vocab", [15, 1000, 2049, 41000])
def test_topk_route_edges(llrs, backend, tmp_path, vocab, spread):
    rng = np.random.default_rng(vocab)
    w = {"normal": rng.standard_normal(vocab) * 3, "five_levels": rng.integers(0, 5, vocab) * 0.7 - 1.4,
         "equal": np.ones(vocab)}[spread].astype(np.float32)
    kv = planted(llrs, backend, tmp_path, w)
    lg = kv.logits()
    edges = {int(np.ceil(vocab / g)) * 9 // 10 for g in (16, 64, 256, 1024)}
    ks = sorted(k for k in {0, 1, 2, 40, 64, 65, vocab - 1, vocab} | edges | {e + 1 for e in edges} if 0 <= k <= vocab)
    checked = 0
    for k in ks:
        for t, tp, pen, n_recent in ((0.0, 1.0, 1.1, 64), (0.7, 0.93, 1.1, 17), (1.3, 1.0, 1.05, 300)):
            recent = rng.integers(0, vocab, n_recent).astype(np.uint32)
            if t > 0 and tp < 1.0 and near_cutoff(lg, t, k, tp, pen, recent):
                continue
            opts = llrs.SamplingOptions(temperature=t, top_p=tp, top_k=k, repetition_penalty=pen)
            for u in (0.0003, 0.377, 0.9991):
                want, margin = f64_sample(lg, t, k, tp, np.float64(np.float32(pen)), recent, u)
                if margin < 1e-5:
                    continue
                got = kv.sample(opts, u, recent)
                assert got == want, (vocab, spread, k, t, tp, pen, n_recent, u)
                checked += 1
    print(f"[topk] vocab {vocab} {spread}: k {ks}, {checked} draws", flush=True)
    assert checked > 30
