"""The work this framework is used for, as cases that can be timed and checked.

A case is a dict of plain values; "op" names the entry points it calls:

  layer     the seven matrix-vector products of one decoder layer, each through
            KernelBackend::matvec's two forms: llrs_matvec_dev on device
            buffers, or HipBackend.matvec on host arrays (host: True)
  matvec    one such product
  prefill   HipQwen2Model.prefill of a prompt, or of a follow-up that starts
            behind rows the cache holds, then the last token's logits
  decode    HipQwen2Model.forward_token, one call a token, as a program does
            that picks each token itself, then the last logits
  sample    KVCache.sample draws over one step's logits

Weights of the model cases come from SynthConfig (normal weights through the
load-time quantizers) or, for the unquantized ones, from a BF16 / F16
checkpoint directory; those of the products are blocks with the codes and
scales such a quantizer leaves.  Shapes are those of bench.py's configs.  The
model cases that stand for one part of a model (a prefill's layers) have a few
of its layers and a small vocabulary, so that the layers are what counts.
"""
import ctypes
import importlib.util
import json
import math
import os
import pathlib
import shutil
import struct
import sys
import tempfile

import numpy as np
import torch

ROOT = pathlib.Path(__file__).resolve().parents[1]

# hidden, intermediate, heads, KV heads, layers, vocabulary
SHAPES = {
    "0.5b": (896, 4864, 14, 2, 24, 151936),
    "1.5b": (1536, 8960, 12, 2, 28, 151936),
    "7b": (3584, 18944, 28, 4, 28, 152064),
}
BLOCK = {"F32": 1, "F16": 1, "BF16": 1, "Q4_0": 32, "Q5_0": 32, "Q8_0": 32, "Q4K": 256, "Q6K": 256}
SIZE = {"F32": 4, "F16": 2, "BF16": 2, "Q4_0": 18, "Q5_0": 22, "Q8_0": 34, "Q4K": 144, "Q6K": 210}
GGML = {0: "F32", 1: "F16", 30: "BF16", 2: "Q4_0", 6: "Q5_0", 8: "Q8_0", 12: "Q4K", 14: "Q6K"}
EPS, THETA = 1e-6, 1e6
CONTEXT = 4096


def listed():
    return [
        # The smallest calls: a 0.5B model's layer, where launches count.
        {"name": "layer_0.5b_q4km", "op": "layer", "shape": "0.5b", "recipe": "q4km", "host": False},
        # The same of a 7B model, 150 MB of weights: the bandwidth of each product.
        {"name": "layer_7b_q4km", "op": "layer", "shape": "7b", "recipe": "q4km", "host": False},
        # The reference's own boundary, host slices in and out.
        {"name": "layer_1.5b_q4k_host", "op": "layer", "shape": "1.5b", "recipe": "q4k", "host": True},
        # Interactive decoding draws each token with the engine's defaults.
        {"name": "sample_defaults", "op": "sample", "vocab": 152064, "draws": 8, "temperature": 0.7, "top_p": 0.9,
         "top_k": 40, "penalty": 1.1, "window": 64},
        # A chat answer of a small model, early in the conversation.
        {"name": "decode_0.5b_q4km", "op": "decode", "shape": "0.5b", "recipe": "q4km", "layers": 24,
         "vocab": 151936, "pos": 128, "steps": 16},
        # The benchmark's model and depth.
        {"name": "decode_7b_q4km", "op": "decode", "shape": "7b", "recipe": "q4km", "layers": 28, "vocab": 152064,
         "pos": 512, "steps": 16},
        # A long conversation, where the cache's rows count too.
        {"name": "decode_1.5b_q4k_deep", "op": "decode", "shape": "1.5b", "recipe": "q4k", "layers": 28,
         "vocab": 151936, "pos": 4000, "steps": 16},
        # An unquantized checkpoint, as it was published.
        {"name": "decode_1.5b_bf16", "op": "decode", "shape": "1.5b", "recipe": "bf16", "layers": 4, "vocab": 32000,
         "pos": 200, "steps": 16},
        # One short question in a chat.
        {"name": "prefill_7b_24", "op": "prefill", "shape": "7b", "recipe": "q4km", "layers": 4, "vocab": 4096,
         "start": 0, "tokens": 24},
        # The benchmark's prompt.
        {"name": "prefill_7b_512", "op": "prefill", "shape": "7b", "recipe": "q4km", "layers": 4, "vocab": 4096,
         "start": 0, "tokens": 512},
        # A document pasted into the context.
        {"name": "prefill_1.5b_4000", "op": "prefill", "shape": "1.5b", "recipe": "q4k", "layers": 4, "vocab": 4096,
         "start": 0, "tokens": 4000},
        # A follow-up of odd length to an earlier turn, unquantized.
        {"name": "prefill_0.5b_bf16_301", "op": "prefill", "shape": "0.5b", "recipe": "bf16", "layers": 4,
         "vocab": 4096, "start": 411, "tokens": 301},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    op = rng.choice(["layer", "matvec", "matvec", "prefill", "prefill", "prefill", "prefill", "decode", "decode",
                     "sample"])
    if op == "layer":
        return {"op": op, "shape": rng.choice(sorted(SHAPES)), "recipe": rng.choice(["q4km", "q4k", "bf16"]),
                "host": rng.random() < 0.3}
    if op == "matvec":
        ty = rng.choice(["Q4_0", "Q5_0", "Q8_0", "Q4K", "Q6K", "F16", "BF16"])
        step = 256 if BLOCK[ty] == 256 else 64
        cols = max(step, _log(rng, 256, 18944) // step * step)
        rows = min(_log(rng, 64, 152064), 152064 * 3584 // cols)
        return {"op": op, "type": ty, "rows": rows, "cols": cols, "host": rng.random() < 0.2}
    if op == "sample":
        return {"op": op, "vocab": _log(rng, 1000, 152064), "draws": rng.randint(2, 8),
                "temperature": rng.choice([0.0, 0.3, 0.7, 1.0, 1.3]), "top_p": rng.choice([0.5, 0.9, 0.95, 1.0]),
                "top_k": rng.choice([0, 1, 20, 40, 100, 1000]), "penalty": rng.choice([1.0, 1.05, 1.1]),
                "window": rng.choice([0, 1, 17, 64, 256])}
    shape = rng.choice(sorted(SHAPES))
    recipe = rng.choice(["q4km", "q4km", "q4k", "bf16", "f16"])
    layers, vocab = rng.randint(2, 4), rng.choice([1000, 4096, 32000])
    if op == "decode":
        return {"op": op, "shape": shape, "recipe": recipe, "layers": layers, "vocab": vocab,
                "pos": _log(rng, 1, 4000), "steps": rng.randint(1, 16)}
    start = rng.choice([0, 0, _log(rng, 1, 2000)])
    return {"op": op, "shape": shape, "recipe": recipe, "layers": layers, "vocab": vocab, "start": start,
            "tokens": _log(rng, 2, 1000 if shape == "7b" else 2000)}


# ------------------------------------------------------------------ the framework

_state = {}


def _package():
    if "llama_rs_amd" not in sys.modules:
        pkg = ROOT / "llama.rs_amd"
        spec = importlib.util.spec_from_file_location("llama_rs_amd", pkg / "__init__.py",
                                                      submodule_search_locations=[str(pkg)])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["llama_rs_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["llama_rs_amd"]


def _backend():
    """A program's one backend."""
    if "backend" not in _state:
        _state["backend"] = _package().HipBackend(0)
    return _state["backend"]


# ------------------------------------------------------------------ inputs

def _generator(seed, device="cuda"):
    g = torch.Generator(device=device)
    g.manual_seed(int(seed) * 1000003 + 12345)
    return g


def _recipe_type(recipe, which, cols):
    """The type the load-time recipe gives a matrix (src/loader.rs:406-447)."""
    if recipe in ("bf16", "f16"):
        return recipe.upper()
    want = "Q4K"
    if recipe == "q4km":
        want = {"v": "Q8_0", "down": "Q6K", "embed": "Q8_0", "head": "Q8_0"}.get(which, "Q4K")
    if BLOCK[want] == 256 and cols % 256:
        want = "Q5_0" if want == "Q4K" else "Q8_0"
    return want


def _layer_matrices(shape, recipe):
    """(type, rows, cols) of a layer's seven matrices, in the order a layer uses them."""
    H, F, nh, nkv = SHAPES[shape][:4]
    kv = H // nh * nkv
    dims = [("q", H, H), ("k", kv, H), ("v", kv, H), ("o", H, H), ("gate", F, H), ("up", F, H), ("down", H, F)]
    return [(_recipe_type(recipe, w, c), r, c) for w, r, c in dims]


def _f16_bytes(x):
    return x.to(torch.float16).view(torch.uint8)


def _random_blocks(ty, rows, cols, g):
    """Native bytes of a [rows, cols] matrix of N(0, 0.02) weights (a cuda
    uint8 tensor [rows, row bytes]): bell-shaped codes and, per block, the
    scale such weights have, give or take a fifth."""
    def normal(*shape):
        return torch.randn(shape, generator=g, device="cuda")

    if ty in ("F16", "BF16"):
        w = normal(rows, cols) * 0.02
        return w.to(torch.float16 if ty == "F16" else torch.bfloat16).view(torch.uint8).reshape(rows, -1)
    bs = BLOCK[ty]
    n = rows * cols // bs
    wobble = 1.0 + 0.2 * (torch.rand((n, 1), generator=g, device="cuda") - 0.5)
    if ty == "Q8_0":
        q = (normal(n, 32) * 52).round_().clamp_(-127, 127).to(torch.int8).view(torch.uint8)
        out = torch.cat([_f16_bytes(0.02 / 52 * wobble), q], 1)
    elif ty in ("Q4_0", "Q5_0"):
        half, sd = (8, 3.2) if ty == "Q4_0" else (16, 6.5)
        q = (normal(n, 32) * sd).round_().clamp_(-half, half - 1).to(torch.int32) + half
        qs = ((q[:, :16] & 15) | ((q[:, 16:] & 15) << 4)).to(torch.uint8)
        parts = [_f16_bytes(0.02 / sd * wobble)]
        if ty == "Q5_0":
            bits = torch.arange(8, device="cuda")
            parts.append(((q >> 4).reshape(n, 4, 8) << bits).sum(2).to(torch.uint8))
        out = torch.cat(parts + [qs], 1)
    elif ty == "Q4K":
        # w = d sc q - dmin m; q around 7.5, so dmin m = 7.5 d sc.
        q = (7.5 + normal(n, 4, 2, 32) * 3.0).round_().clamp_(0, 15).to(torch.int32)
        qs = (q[:, :, 0] | (q[:, :, 1] << 4)).reshape(n, 128).to(torch.uint8)
        sc = torch.randint(38, 64, (n, 8), generator=g, device="cuda", dtype=torch.int32)
        mn = (sc + torch.randint(-2, 3, (n, 8), generator=g, device="cuda", dtype=torch.int32)).clamp_(0, 63)
        lo = torch.cat([(sc[:, :4] | ((sc[:, 4:] >> 4) << 6)), (mn[:, :4] | ((mn[:, 4:] >> 4) << 6)),
                        ((sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4))], 1).to(torch.uint8)
        d = 0.02 / (3.0 * 50) * wobble
        out = torch.cat([_f16_bytes(d), _f16_bytes(7.5 * d), lo, qs], 1)
    elif ty == "Q6K":
        q = (32 + normal(n, 2, 4, 32) * 13).round_().clamp_(0, 63).to(torch.int32)  # [half][quarter][32]
        ql = torch.cat([(q[:, :, 0] & 15) | ((q[:, :, 2] & 15) << 4), (q[:, :, 1] & 15) | ((q[:, :, 3] & 15) << 4)], 2)
        qh = (q[:, :, 0] >> 4) | ((q[:, :, 1] >> 4) << 2) | ((q[:, :, 2] >> 4) << 4) | ((q[:, :, 3] >> 4) << 6)
        sc = torch.randint(70, 128, (n, 16), generator=g, device="cuda", dtype=torch.int32)
        sc = torch.where(torch.rand((n, 16), generator=g, device="cuda") < 0.5, sc, -sc).to(torch.int8)
        out = torch.cat([ql.reshape(n, 128).to(torch.uint8), qh.reshape(n, 64).to(torch.uint8),
                         sc.view(torch.uint8), _f16_bytes(0.02 / (13 * 99) * wobble)], 1)
    else:
        raise ValueError(ty)
    return out.reshape(rows, -1)


def _matrices(case):
    return _layer_matrices(case["shape"], case["recipe"]) if case["op"] == "layer" else [
        (case["type"], case["rows"], case["cols"])]


def _activation(cols, g):
    """Activations with the heavy channels a decoder's have."""
    x = torch.randn((cols,), generator=g, device="cuda")
    return x * torch.where(torch.rand((cols,), generator=g, device="cuda") < 0.01, 8.0, 1.0)


def _prepare_products(case, seed):
    P, be, g = _package(), _backend(), _generator(seed)
    calls = []
    for ty, rows, cols in _matrices(case):
        data = _random_blocks(ty, rows, cols, g).cpu().numpy().tobytes()
        w = be.upload(P.QuantTensor.from_owned(data, (rows, cols), P.QuantType[ty]))
        x, y = _activation(cols, g), torch.zeros(rows, device="cuda")
        if case["host"]:
            x, y = x.cpu().numpy(), y.cpu().numpy()
        calls.append((w, x, y))
    torch.cuda.synchronize()
    return {"case": case, "backend": be, "calls": calls, "matvec_dev": P.lib().llrs_matvec_dev}


def _tokens(n, vocab, seed):
    return np.random.default_rng(seed).integers(0, vocab, n).astype(np.uint32)


def _float_weights(case, seed):
    """Name -> tensor of an unquantized checkpoint, in the published names."""
    H, F, nh, nkv = SHAPES[case["shape"]][:4]
    kv, ty = H // nh * nkv, torch.bfloat16 if case["recipe"] == "bf16" else torch.float16
    g, out = _generator(seed), {}

    def normal(name, *shape, base=0.0):
        out[name] = (base + 0.02 * torch.randn(shape, generator=g, device="cuda")).to(ty)

    normal("model.embed_tokens.weight", case["vocab"], H)
    for i in range(case["layers"]):
        p = "model.layers.%d." % i
        normal(p + "input_layernorm.weight", H, base=1.0)
        normal(p + "post_attention_layernorm.weight", H, base=1.0)
        for w, rows in (("q", H), ("k", kv), ("v", kv)):
            normal(p + "self_attn.%s_proj.weight" % w, rows, H)
            normal(p + "self_attn.%s_proj.bias" % w, rows)
        normal(p + "self_attn.o_proj.weight", H, H)
        normal(p + "mlp.gate_proj.weight", F, H)
        normal(p + "mlp.up_proj.weight", F, H)
        normal(p + "mlp.down_proj.weight", H, F)
    normal("model.norm.weight", H, base=1.0)
    normal("lm_head.weight", case["vocab"], H)
    return out


def _write_checkpoint(case, seed, folder):
    H, F, nh, nkv = SHAPES[case["shape"]][:4]
    with open(os.path.join(folder, "config.json"), "w") as f:
        json.dump({"model_type": "qwen2", "hidden_size": H, "intermediate_size": F, "num_attention_heads": nh,
                   "num_key_value_heads": nkv, "num_hidden_layers": case["layers"], "vocab_size": case["vocab"],
                   "max_position_embeddings": 32768, "rms_norm_eps": EPS, "rope_theta": THETA,
                   "tie_word_embeddings": False}, f)
    weights, header, at = _float_weights(case, seed), {}, 0
    for name, t in weights.items():
        n = t.numel() * 2
        header[name] = {"dtype": case["recipe"].upper(), "shape": list(t.shape), "data_offsets": [at, at + n]}
        at += n
    text = json.dumps(header).encode()
    text += b" " * (-len(text) % 8)
    with open(os.path.join(folder, "model.safetensors"), "wb") as f:
        f.write(struct.pack("<Q", len(text)) + text)
        for t in weights.values():
            f.write(t.view(torch.int16).cpu().numpy().tobytes())


def _model(case, seed):
    P, be = _package(), _backend()
    H, F, nh, nkv = SHAPES[case["shape"]][:4]
    if case["recipe"] in ("bf16", "f16"):
        folder = tempfile.mkdtemp(prefix="cases_")
        try:
            _write_checkpoint(case, seed, folder)
            return P.ModelLoader.load(folder, be)
        finally:
            shutil.rmtree(folder)
    recipe = {"q4km": P.LoadQuantization.Q4KM, "q4k": P.LoadQuantization.Q4K}[case["recipe"]]
    return P.HipQwen2Model.synthetic(be, P.SynthConfig(
        H, F, nh, nkv, case["layers"], case["vocab"], rms_norm_eps=EPS, rope_theta=THETA,
        tie_word_embeddings=case["shape"] != "7b", recipe=recipe, seed=seed))


def _model_tokens(case, seed):
    """(tokens the cache holds before the pass, tokens of the pass)"""
    before, now = (case["pos"], case["steps"]) if case["op"] == "decode" else (case["start"], case["tokens"])
    t = _tokens(before + now, case["vocab"], seed)
    return t[:before], t[before:]


def _sample_inputs(case, seed):
    r = np.random.default_rng(seed)
    return r.random(case["draws"], dtype=np.float32), r.integers(0, case["vocab"], case["window"]).astype(np.uint32)


def prepare(case, seed):
    P = _package()
    if case["op"] in ("layer", "matvec"):
        return _prepare_products(case, seed)
    if case["op"] == "sample":
        # A one-layer model of this vocabulary; its logits are as spread as a model's.
        model = P.HipQwen2Model.synthetic(_backend(), P.SynthConfig(
            896, 256, 14, 2, 1, case["vocab"], rms_norm_eps=EPS, rope_theta=THETA, tie_word_embeddings=False,
            weight_std=0.05, seed=seed))
        kv = P.KVCache(model, 64)
        model.prefill(_tokens(8, case["vocab"], seed), 0, kv)
        draws, window = _sample_inputs(case, seed)
        opts = P.SamplingOptions(case["temperature"], case["top_p"], case["top_k"], case["penalty"])
        return {"case": case, "kv": kv, "opts": opts, "draws": draws, "window": window}
    model = _model(case, seed)
    kv = P.KVCache(model, CONTEXT)
    before, now = _model_tokens(case, seed)
    if len(before):
        model.prefill(before, 0, kv)
    return {"case": case, "model": model, "kv": kv, "before": len(before), "tokens": now,
            "compute": P.LogitsMode.COMPUTE}


# ------------------------------------------------------------------ one pass

def run(state):
    case = state["case"]
    if case["op"] in ("layer", "matvec"):
        be = state["backend"]
        if case["host"]:
            for w, x, y in state["calls"]:
                be.matvec(w, x, y)
        else:
            for w, x, y in state["calls"]:
                if state["matvec_dev"](be.handle, w.handle, ctypes.c_void_p(x.data_ptr()),
                                       ctypes.c_void_p(y.data_ptr())):
                    raise RuntimeError("llrs_matvec_dev failed")
        return [y for _, _, y in state["calls"]]
    if case["op"] == "sample":
        return [state["kv"].sample(state["opts"], u, state["window"]) for u in state["draws"]]
    if case["op"] == "prefill":
        state["model"].prefill(state["tokens"], state["before"], state["kv"])
    else:
        for i, t in enumerate(state["tokens"]):
            state["model"].forward_token(int(t), state["before"] + i, state["kv"], state["compute"])
    return {"logits": state["kv"].logits()}


# ------------------------------------------------------------------ what a pass cannot do without

def _nbytes(ty, rows, cols):
    return rows * cols // BLOCK[ty] * SIZE[ty]


def work(case):
    if case["op"] in ("layer", "matvec"):
        m = _matrices(case)
        return {"bytes": sum(_nbytes(*w) + 4 * (w[1] + w[2]) for w in m), "flops": sum(2 * r * c for _, r, c in m)}
    if case["op"] == "sample":
        return {"bytes": case["draws"] * 4 * case["vocab"], "flops": case["draws"] * 4 * case["vocab"]}
    H, F, nh, nkv = SHAPES[case["shape"]][:4]
    kv, L, V = H // nh * nkv, case["layers"], case["vocab"]
    m = _layer_matrices(case["shape"], case["recipe"])
    weights, params = L * sum(_nbytes(*w) for w in m), L * sum(r * c for _, r, c in m)
    head = _nbytes(_recipe_type(case["recipe"], "head", H), V, H)
    before, n = (case["pos"], case["steps"]) if case["op"] == "decode" else (case["start"], case["tokens"])
    seen = sum(range(before + 1, before + n + 1))  # positions attended, over the tokens
    flops = 2 * params * n + 4 * L * H * seen
    if case["op"] == "decode":  # each step reads the weights, the head and the rows so far
        return {"bytes": n * (weights + head + 4 * V) + 8 * L * kv * (seen + n), "flops": flops + 2 * V * H * n}
    return {"bytes": weights + head + 4 * V + 8 * L * kv * (before + n), "flops": flops + 2 * V * H}


def tolerance(case):
    if case["op"] == "sample":
        return "exact"
    # Four times the error against 64 bits that these paths show.
    floats = case.get("recipe") in ("bf16", "f16") or case.get("type") in ("F16", "BF16")
    if case["op"] in ("layer", "matvec"):
        # 15-bit activation digits for the quantized types (5.5e-5 off), f32 sums otherwise (2.3e-7).
        return {"rel": 1e-6 if floats else 2e-4}
    # Logits at the end of a stack, whose roundings travel through every layer: f32 sums (2.4e-6 off),
    # or digits in every product of a decode step (3.6e-4) and in the head alone of a prefill (3.8e-5).
    if floats:
        return {"rel": 1e-5}
    return {"rel": 1.5e-3 if case["op"] == "decode" else 2e-4}


# ------------------------------------------------------------------ in 64 bits

def _dequant(ty, b, rows, cols):
    """float64 values of native rows (a cuda uint8 tensor of rows * row bytes)."""
    if ty in ("F32", "F16", "BF16"):
        t = {"F32": torch.float32, "F16": torch.float16, "BF16": torch.bfloat16}[ty]
        return b.reshape(-1).view(t).to(torch.float64).reshape(rows, cols)
    b = b.reshape(-1, SIZE[ty])
    n = b.shape[0]

    def f16(at):
        return b[:, at:at + 2].contiguous().view(torch.float16).to(torch.float64)

    def ints(x):
        return x.to(torch.int32)

    if ty == "Q8_0":
        v = f16(0) * b[:, 2:].contiguous().view(torch.int8).to(torch.float64)
    elif ty == "Q4_0":
        q = ints(b[:, 2:])
        v = f16(0) * (torch.cat([q & 15, q >> 4], 1) - 8).to(torch.float64)
    elif ty == "Q5_0":
        q, bits = ints(b[:, 6:]), torch.arange(8, device=b.device)
        high = ((ints(b[:, 2:6]).unsqueeze(2) >> bits) & 1).reshape(n, 32)
        v = f16(0) * ((torch.cat([q & 15, q >> 4], 1) | (high << 4)) - 16).to(torch.float64)
    elif ty == "Q4K":
        s = ints(b[:, 4:16])
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1)
        q = ints(b[:, 16:]).reshape(n, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 2).reshape(n, 8, 32)
        v = (f16(0) * sc.to(torch.float64)).unsqueeze(2) * q - (f16(2) * mn.to(torch.float64)).unsqueeze(2)
    elif ty == "Q6K":
        ql, qh = ints(b[:, :128]).reshape(n, 2, 2, 32), ints(b[:, 128:192]).reshape(n, 2, 1, 32)
        low = torch.cat([ql & 15, ql >> 4], 2)
        high = (qh >> (2 * torch.arange(4, device=b.device)).reshape(1, 1, 4, 1)) & 3
        sc = b[:, 192:208].contiguous().view(torch.int8).to(torch.float64).reshape(n, 2, 4, 2, 1)
        v = f16(208).reshape(n, 1, 1, 1, 1) * sc * ((low | (high << 4)) - 32).reshape(n, 2, 4, 2, 16)
    else:
        raise ValueError(ty)
    return v.reshape(rows, cols)


def _read_gguf(path):
    """Name -> (type, rows, cols, bytes) of a GGUF v3 file."""
    raw = np.memmap(path, dtype=np.uint8, mode="r")
    at = 24

    def take(fmt):
        nonlocal at
        v = struct.unpack_from("<" + fmt, raw, at)
        at += struct.calcsize("<" + fmt)
        return v[0] if len(v) == 1 else v

    def text():
        nonlocal at
        n = take("Q")
        at += n
        return bytes(raw[at - n:at]).decode()

    ntensors, nkv = struct.unpack_from("<QQ", raw, 8)
    for _ in range(nkv):
        text()
        kind = take("I")
        if kind == 8:
            text()
        else:
            take({4: "I", 5: "i", 6: "f", 10: "Q"}[kind])
    infos = []
    for _ in range(ntensors):
        name, nd = text(), take("I")
        dims = [take("Q") for _ in range(nd)]
        infos.append((name, GGML[take("I")], dims, take("Q")))
    base = (at + 31) // 32 * 32
    out = {}
    for name, ty, dims, off in infos:
        rows, cols = (dims[1], dims[0]) if len(dims) == 2 else (1, dims[0])
        out[name] = (ty, rows, cols, raw[base + off:base + off + _nbytes(ty, rows, cols)])
    return out


def _exact_logits(case, seed, get, rows_of):
    """Last-token logits in float64: get(name) is a matrix or vector,
    rows_of(name, ids) some rows of one; names as in a GGUF file."""
    H, F, nh, nkv = SHAPES[case["shape"]][:4]
    hd, f64 = H // nh, torch.float64
    ids = np.concatenate(_model_tokens(case, seed))
    T = len(ids)
    x = rows_of("token_embd.weight", ids)
    # The angles are float32, as the model defines them (src/model.rs:76-84).
    half = hd // 2
    inv = np.float32(1) / np.power(np.float32(THETA), np.float32(2) * np.arange(half, dtype=np.float32) / np.float32(hd))
    ang = torch.from_numpy(np.arange(T, dtype=np.float32)[:, None] * inv[None]).cuda().to(f64)
    cos, sin = ang.cos().unsqueeze(1), ang.sin().unsqueeze(1)

    def norm(v, name):
        return v / torch.sqrt((v * v).mean(1, keepdim=True) + EPS) * get(name).reshape(1, -1)

    def rope(v):
        a, b = v[:, :, :half], v[:, :, half:]
        return torch.cat([a * cos - b * sin, a * sin + b * cos], 2)

    mask = torch.triu(torch.full((T, T), -math.inf, device="cuda", dtype=f64), 1)
    for i in range(case["layers"]):
        p = "blk.%d." % i
        h = norm(x, p + "attn_norm.weight")
        q, k, v = (h @ get(p + "attn_%s.weight" % w).T + get(p + "attn_%s.bias" % w).reshape(1, -1) for w in "qkv")
        q, k, v = rope(q.reshape(T, nh, hd)), rope(k.reshape(T, nkv, hd)), v.reshape(T, nkv, hd)
        heads = []
        for j in range(nh):
            s = q[:, j] @ k[:, j * nkv // nh].T / math.sqrt(hd) + mask
            heads.append(torch.softmax(s, 1) @ v[:, j * nkv // nh])
        x = x + torch.cat(heads, 1) @ get(p + "attn_output.weight").T
        h = norm(x, p + "ffn_norm.weight")
        g = h @ get(p + "ffn_gate.weight").T
        x = x + (g * torch.sigmoid(g) * (h @ get(p + "ffn_up.weight").T)) @ get(p + "ffn_down.weight").T
    h = norm(x[-1:], "output_norm.weight")
    parts = [h @ rows_of("head", np.arange(a, min(case["vocab"], a + 16384))).T
             for a in range(0, case["vocab"], 16384)]
    return {"logits": torch.cat(parts, 1).reshape(-1).cpu().numpy()}


_HF = {"attn_norm": "input_layernorm", "ffn_norm": "post_attention_layernorm", "attn_q": "self_attn.q_proj",
       "attn_k": "self_attn.k_proj", "attn_v": "self_attn.v_proj", "attn_output": "self_attn.o_proj",
       "ffn_gate": "mlp.gate_proj", "ffn_up": "mlp.up_proj", "ffn_down": "mlp.down_proj"}


def _exact_model(case, seed):
    if case["recipe"] in ("bf16", "f16"):
        weights = _float_weights(case, seed)

        def find(name):
            if name.startswith("blk."):
                _, i, w, kind = name.split(".")
                return weights["model.layers.%s.%s.%s" % (i, _HF[w], kind)]
            return weights[{"token_embd.weight": "model.embed_tokens.weight", "output_norm.weight": "model.norm.weight",
                            "head": "lm_head.weight"}[name]]

        return _exact_logits(case, seed, lambda n: find(n).to(torch.float64),
                             lambda n, ids: find(n)[torch.from_numpy(ids.astype(np.int64)).cuda()].to(torch.float64))
    folder = tempfile.mkdtemp(prefix="cases_")
    try:
        path = os.path.join(folder, "model.gguf")
        _model(case, seed).export_gguf(path)
        t = _read_gguf(path)
        t["head"] = t.get("output.weight", t["token_embd.weight"])

        def get(name):
            ty, rows, cols, b = t[name]
            return _dequant(ty, torch.from_numpy(np.array(b)).cuda(), rows, cols)

        def rows_of(name, ids):
            ty, rows, cols, b = t[name]
            sub = np.ascontiguousarray(b.reshape(rows, -1)[ids])
            return _dequant(ty, torch.from_numpy(sub).cuda(), len(ids), cols)

        return _exact_logits(case, seed, get, rows_of)
    finally:
        shutil.rmtree(folder)


def _exact_sample(case, seed):
    """The draws by their definition (src/engine.rs:253-325) on the step's logits."""
    state = prepare(case, seed)
    v = state["kv"].logits().astype(np.float64)
    if case["penalty"] != 1.0:
        w = np.unique(state["window"])
        v[w] = np.where(v[w] > 0, v[w] / np.float32(case["penalty"]), v[w] * np.float32(case["penalty"]))
    if case["temperature"] > 0:
        v /= np.float32(case["temperature"])
    order = np.argsort(-v, kind="stable")
    if case["temperature"] <= 0:
        return [int(order[0])] * case["draws"]
    order = order[:case["top_k"] or None]
    p = np.exp(v[order] - v[order[0]])
    c = np.cumsum(p / p.sum())
    kept = min(len(c), int(np.searchsorted(c, float(np.float32(case["top_p"])))) + 1)
    return [int(order[min(kept - 1, int(np.searchsorted(c[:kept], float(u) * c[kept - 1])))]) for u in state["draws"]]


def exact(case, seed):
    if case["op"] in ("layer", "matvec"):
        g, out = _generator(seed), []
        for ty, rows, cols in _matrices(case):
            b = _random_blocks(ty, rows, cols, g)
            x = _activation(cols, g).to(torch.float64)
            step = max(1, (1 << 27) // cols)
            y = torch.cat([_dequant(ty, b[r:r + step], min(step, rows - r), cols) @ x for r in range(0, rows, step)])
            out.append(y.cpu().numpy() if case["host"] else y)
        return out
    if case["op"] == "sample":
        return _exact_sample(case, seed)
    if case["shape"] == "7b" and case["layers"] > 4:
        return None  # a 4.7 GB export, and every matrix in 64 bits: too long
    return _exact_model(case, seed)
