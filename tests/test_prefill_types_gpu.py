"""Batched prefill per weight type and token count vs the CPU oracle (MI355X).

Tolerances: activations and weights meet as 22-bit f16 pairs and f32 sums, so
a product is off by about 1e-6 of its magnitude; logits of these two-layer
models (order 1) may be off by 2e-4 (the quantized LM head's 15-bit activation
digits among it) and K/V rows (order 1) by 2e-5.
"""
from __future__ import annotations

import numpy as np
import pytest

from hf_checkpoint import write_checkpoint

pytestmark = pytest.mark.gpu


def check(llrs, oracle, model, tmp_path, vocab, layers, n, seed):
    model.export_gguf(tmp_path / "m.gguf")
    om = oracle.load(tmp_path / "m.gguf")
    om.new_state(n + 4)
    kv = llrs.KVCache(model, n + 4)
    prompt = np.random.default_rng(seed).integers(0, vocab, n).astype(np.uint32)
    model.prefill(prompt, 0, kv)
    om.prefill(prompt, 0)
    err = float(np.abs(kv.logits() - om.logits()).max())
    print(f"[types] n={n} logits max-abs err {err:.3e}", flush=True)
    assert err <= 2e-4 * max(1.0, float(np.abs(om.logits()).max()))
    for layer in range(layers):
        for which in ("k", "v"):
            a, b = kv.layer(layer, which, n), om.kv(layer, which, n)
            assert float(np.abs(a - b).max()) <= 2e-5 * max(1.0, float(np.abs(b).max())), (layer, which)


@pytest.mark.parametrize("n", [2, 65, 257], ids=["2", "65", "257"])
@pytest.mark.parametrize("dtype", ["BF16", "F16", "F32"])
@pytest.mark.parametrize("staged", [False, True], ids=["default", "lds_staged"])
def test_prefill_float_weights(llrs, backend, oracle, tmp_path, monkeypatch, dtype, n, staged):
    """Unquantized checkpoints: FFN matrices of 2,080 rows (sixteen 128-row
    tiles and a remainder), two tokens, one past a 64-token tile, one past
    two 128-token tiles; on the default route and on the LDS-staged kernel
    that large 16-bit products take."""
    if staged:
        monkeypatch.setenv("LLRS_PREFILL_CODES", "f32")
    cfg = llrs.SynthConfig(hidden_size=256, intermediate_size=2080, num_attention_heads=4, num_key_value_heads=2,
                           num_hidden_layers=2, vocab_size=1000, max_position_embeddings=512, seed=51,
                           tie_word_embeddings=False)
    write_checkpoint(llrs, cfg, tmp_path / "ck", dtype)
    model = llrs.ModelLoader.load(tmp_path / "ck", backend)
    check(llrs, oracle, model, tmp_path, cfg.vocab_size, cfg.num_hidden_layers, n, 51 + n)


@pytest.mark.parametrize("n", [2, 16, 17, 32, 33, 65, 130])
@pytest.mark.parametrize("hidden,heads,ffn,recipe", [(512, 4, 2304, "Q4KM"), (512, 8, 2112, "Q4K"),
                                                     (352, 11, 2112, "Q4KM"), (384, 6, 2112, "Q4K")],
                         ids=["q4k_q8_q6k", "q4k_q5", "q5_q8_ragged_k", "q5"])
def test_prefill_quantized_weights(llrs, backend, oracle, tmp_path, hidden, heads, ffn, recipe, n):
    """The register-decoded products: 16-, 32- and 64-token tiles full, with one
    token too many and with remainders; FFN rows that end inside a row tile
    (2,112); rows of a 32-column remainder past whole steps (352, 2,112); an
    odd number of 256-column blocks (2,304); q/k/v in segments and apart (352
    is no multiple of 128)."""
    cfg = llrs.SynthConfig(hidden_size=hidden, intermediate_size=ffn, num_attention_heads=heads,
                           num_key_value_heads=heads if heads == 11 else 2, num_hidden_layers=2, vocab_size=500,
                           max_position_embeddings=256, seed=57, tie_word_embeddings=False,
                           recipe=getattr(llrs.LoadQuantization, recipe))
    model = llrs.HipQwen2Model.synthetic(backend, cfg)
    check(llrs, oracle, model, tmp_path, cfg.vocab_size, cfg.num_hidden_layers, n, 57 + n)


@pytest.mark.parametrize("hd", [16, 32, 64, 128])
def test_prefill_chunks_and_unaligned_start(llrs, backend, oracle, tmp_path, hd):
    """37 tokens, then 2,063 from position 37: the second call grows the row
    buffers, starts inside a 16-position block of the f16 K/V planes, and runs
    as a 2,048-row chunk and a 15-row one (position 2,085 starts inside a block
    again); in one call of 2,100 the last chunk starts at a block's edge.
    hidden 1,024 with Q4_K o (its sums come from the attention kernel, or from
    a pass of their own at head_dim 16)."""
    cfg = llrs.SynthConfig(hidden_size=1024, intermediate_size=1024, num_attention_heads=1024 // hd,
                           num_key_value_heads=256 // hd, num_hidden_layers=2, vocab_size=500,
                           max_position_embeddings=2304, seed=63, tie_word_embeddings=False)
    model = llrs.HipQwen2Model.synthetic(backend, cfg)
    model.export_gguf(tmp_path / "m.gguf")
    om = oracle.load(tmp_path / "m.gguf")
    om.new_state(2104)
    prompt = np.random.default_rng(63).integers(0, cfg.vocab_size, 2100).astype(np.uint32)
    om.prefill(prompt, 0)
    for cut in (37, 0):
        kv = llrs.KVCache(model, 2104)
        if cut:
            model.prefill(prompt[:cut], 0, kv)
        model.prefill(prompt[cut:], cut, kv)
        err = float(np.abs(kv.logits() - om.logits()).max())
        print(f"[chunks] hd={hd} cut={cut} logits max-abs err {err:.3e}", flush=True)
        assert err <= 2e-4 * max(1.0, float(np.abs(om.logits()).max()))
        for layer in range(cfg.num_hidden_layers):
            for which in ("k", "v"):
                a, b = kv.layer(layer, which, 2100), om.kv(layer, which, 2100)
                assert float(np.abs(a - b).max()) <= 2e-5 * max(1.0, float(np.abs(b).max())), (layer, which)
