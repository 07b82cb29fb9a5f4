"""Products of F32 / F16 / BF16 weights, alone and in a decode step (MI355X).

A lane adds at most cols / 64 terms and six levels of a tree follow, in f32:
an output is off by at most (cols / 64 + 8) * 2^-24 of the sum of its terms'
magnitudes.  A decode step chains five such products a layer and their norms;
its logits (order 1) may be off by 5e-5, the H-term bounds of two layers' chain
at 4,352 columns, 4 * 2 * 76 * 2^-24, rounded up.
"""
from __future__ import annotations

import numpy as np
import pytest

from hf_checkpoint import write_checkpoint

pytestmark = pytest.mark.gpu

TYPES = {"F32": 0, "F16": 1, "BF16": 30}


@pytest.mark.parametrize("rows,cols", [(1, 8), (3, 520), (5, 1536), (6, 2048), (9, 2056), (7, 9000), (2, 8960),
                                       (8191, 2056), (8195, 264), (8192, 2056)])
@pytest.mark.parametrize("ty", list(TYPES))
def test_float_products(llrs, backend, ty, rows, cols):
    """The product without a norm, one and four (from 8,192 on) rows a wave: one
    chunk, rows that fill the unrolled loop, end inside it, or in a 16-byte load
    after it; row counts off the workgroups' multiples."""
    rng = np.random.default_rng(rows + cols)
    w = rng.standard_normal((rows, cols)).astype(np.float32)
    if ty == "F16":
        data = w.astype(np.float16)
        w = data.astype(np.float64)
    elif ty == "BF16":
        data = (w.view(np.uint32) >> 16).astype(np.uint16)
        w = (data.astype(np.uint32) << 16).view(np.float32).astype(np.float64)
    else:
        data = w
        w = w.astype(np.float64)
    x = rng.standard_normal(cols).astype(np.float32)
    t = backend.upload(llrs.QuantTensor.from_owned(data.tobytes(), (rows, cols), TYPES[ty]))
    y = np.full(rows, np.nan, np.float32)
    backend.matvec(t, x, y)
    bound = (cols / 64 + 8) * 2.0**-24 * (np.abs(w) @ np.abs(x.astype(np.float64)))
    err = np.abs(y - w @ x.astype(np.float64))
    print(f"[float] {ty} {rows}x{cols} err / bound {float((err / bound).max()):.3f}", flush=True)
    assert (err <= bound).all()


@pytest.mark.parametrize("hidden,heads,kv_heads,ffn,vocab", [(256, 4, 2, 520, 8195), (576, 9, 3, 4104, 300),
                                                             (1088, 17, 1, 9000, 8193), (4352, 34, 2, 264, 300)])
@pytest.mark.parametrize("dtype", list(TYPES))
def test_float_decode_step(llrs, backend, oracle, tmp_path, dtype, hidden, heads, kv_heads, ffn, vocab):
    """The products behind a norm: q/k/v in one launch, gate/up, the LM head; rows
    of 32 to 1,088 chunks (batches of two and four, partly filled, several a
    row), one round and several of a workgroup's waves, a norm over more columns
    than a workgroup's registers hold (4,352), an LM head of whole and ragged
    groups of two and four rows."""
    if hidden == 4352 and dtype != "BF16":
        pytest.skip("one type's weights of this size are enough")
    cfg = llrs.SynthConfig(hidden_size=hidden, intermediate_size=ffn, num_attention_heads=heads,
                           num_key_value_heads=kv_heads, num_hidden_layers=2, vocab_size=vocab,
                           max_position_embeddings=64, seed=71, tie_word_embeddings=False)
    write_checkpoint(llrs, cfg, tmp_path / "ck", dtype)
    model = llrs.ModelLoader.load(tmp_path / "ck", backend)
    model.export_gguf(tmp_path / "m.gguf")
    om = oracle.load(tmp_path / "m.gguf")
    om.new_state(16)
    kv = llrs.KVCache(model, 16)
    prompt = np.random.default_rng(71).integers(0, vocab, 5).astype(np.uint32)
    om.prefill(prompt, 0)
    for i, t in enumerate(prompt):
        model.forward_token(int(t), i, kv)
    err = float(np.abs(kv.logits() - om.logits()).max())
    print(f"[float] {dtype} H={hidden} logits max-abs err {err:.3e}", flush=True)
    assert err <= 5e-5 * max(1.0, float(np.abs(om.logits()).max()))
