"""The work that users of this framework have it do, as cases that can be timed and checked: lazy graphs over rows and long vectors,
products of every type and layout, and the decoders of the registry, prompts and replies.

A case is a dict of plain values.  `prepare` makes what a program has in hand before the call, `run` is one pass through the public
entry points, `exact` says in 64 bits, without this package, what it should give."""
import ctypes
import json
import math
import os
import shutil
import tempfile

import numpy as np
import torch

import ug_amd
from ug_amd import LazyBuffer as LB
from ug_amd import Schedule, st_writer
from ug_amd.graphs import fused_reduce_graph

EPS = 1e-5
TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
UG = {"f32": ug_amd.F32, "f16": ug_amd.F16, "bf16": ug_amd.BF16}


# ---- the cases -------------------------------------------------------------------------------------------------------------------
def listed():
    return [
        # lazy graphs.  The smallest call there is in earnest (one layer's scores of a short sequence): two launches, all latency.
        {"name": "softmax_32x1024", "kind": "rows", "op": "softmax", "rows": 32, "cols": 1024},
        # the norm of a long prompt's rows at the width of the 1.1 B llama
        {"name": "rms_norm_1900x2048", "kind": "rows", "op": "rms_norm", "rows": 1900, "cols": 2048},
        # a large softmax whose rows start at any four-byte address
        {"name": "softmax_16411x1531", "kind": "rows", "op": "softmax", "rows": 16411, "cols": 1531},
        # sum(a * b + 0.5 * a): elementwise work fused into a reduction of the whole tensor, the benchmark's own workload
        {"name": "reduce_16777216", "kind": "reduce", "n": 1 << 24},
        # products: the benchmark's batch in 32 bits, a large one in bf16 against a weight matrix, and a 16-bit one of sizes that nothing divides
        {"name": "bmm_f32_8x1024", "kind": "product", "dtype": "f32", "nt": False, "b": 8, "m": 1024, "n": 1024, "k": 1024},
        {"name": "mm_bf16_4096", "kind": "product", "dtype": "bf16", "nt": True, "b": 1, "m": 4096, "n": 4096, "k": 4096},
        {"name": "mm_f16_ragged", "kind": "product", "dtype": "f16", "nt": False, "b": 1, "m": 1000, "n": 777, "k": 1531},
        # prompts: a document for the llama, a question for the routed experts, a long context for the delta rule
        {"name": "llama_prompt_1900", "kind": "prompt", "design": "llama", "width": 2048, "dtype": "bf16", "prompt": 1900},
        {"name": "tanolorn_prompt_509", "kind": "prompt", "design": "tanolorn", "width": 2048, "dtype": "bf16", "prompt": 509},
        {"name": "tugelorn_prompt_2048", "kind": "prompt", "design": "tugelorn", "width": 2048, "dtype": "bf16", "prompt": 2048},
        # replies: a short prompt and 127 single positions behind it, one at a time, in 32 bits and in bf16
        {"name": "llama_reply_f32", "kind": "reply", "design": "llama", "width": 2048, "dtype": "f32", "prompt": 128, "steps": 127},
        {"name": "tugelorn_reply_bf16", "kind": "reply", "design": "tugelorn", "width": 1024, "dtype": "bf16", "prompt": 100, "steps": 127},
    ]


def _size(rng, lo, hi):
    """A size between lo and hi, even on a logarithmic scale; every second one a multiple of 64 where that can be."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return max(64, n // 64 * 64) if hi >= 64 and n >= 64 and rng.random() < 0.5 else n


def draw(rng):
    kind = rng.choice(["rows", "reduce", "product", "product", "prompt", "prompt", "reply"])
    if kind == "rows":
        cols = _size(rng, 64, 8192)
        return {"kind": kind, "op": rng.choice(["softmax", "rms_norm"]), "rows": _size(rng, 1, min(16411, (1 << 25) // cols)), "cols": cols}
    if kind == "reduce":
        return {"kind": kind, "n": _size(rng, 1 << 10, 1 << 25)}
    if kind == "product":
        b = rng.choice([1, 1, 1, rng.randint(2, 16)])
        dims = {d: _size(rng, 16, 4096) for d in "mnk"}
        while 2 * b * dims["m"] * dims["n"] * dims["k"] > 1.2e11:
            dims[rng.choice("mnk")] //= 2
        return {"kind": kind, "dtype": rng.choice(["f32", "f16", "bf16"]), "nt": rng.random() < 0.5, "b": b, **dims}
    case = {"kind": kind, "design": rng.choice(["llama", "tanolorn", "tugelorn"]), "width": rng.choice([1024, 2048]), "dtype": rng.choice(["bf16", "bf16", "f32"])}
    if kind == "prompt":
        return {**case, "prompt": _size(rng, 16, 2048)}
    if case["design"] == "tanolorn":  # its experts in 32 bits would be more than the largest listed reply reads
        case["dtype"] = "bf16"
    return {**case, "prompt": _size(rng, 16, 512), "steps": rng.randint(100, 127)}


# ---- the models: configurations of the benchmark -----------------------------------------------------------------------------------
VOCAB = 32000


def _config(design, width):
    heads, ff = width // 128, width * 11 // 4
    if design == "llama":
        return {"model_type": "llama", "hidden_size": width, "intermediate_size": ff, "max_position_embeddings": 4096, "num_attention_heads": width // 64, "num_key_value_heads": 4,
                "num_hidden_layers": 6, "rms_norm_eps": EPS, "vocab_size": VOCAB}
    if design == "tugelorn":
        sizes = {"heads": heads, "kv_heads": heads // 4, "dim": 128, "vdim": 128, "scale": 128 ** -0.5}
        window = {"type": "attention", "mixer": {**sizes, "mask": {"size": 1024}, "rot": {"base": 10000.0, "dims": 128, "scaling": {"factor": 2.0}}}}
        full = {"type": "attention_2", "mixer": {**sizes, "q_temp": {"coef": 0.1, "every": 4096}}}
        delta = {"type": "channel_delta", "mixer": {"heads": heads, "kv_heads": heads, "dim": 128, "vdim": 128, "conv": 4}}
        return {"architecture": "Tugelorn", "vocab": VOCAB, "width": width, "norm": {"eps": EPS}, "residual_mult": 0.5,
                "layers": [{**((delta, window, delta, full)[i % 4]), "mlp": {"kind": "dense", "ff": ff, "limit": 7.0}} for i in range(6)]}
    attn = {"heads": heads, "dim": 128, "rot_dim": 64, "vdim": 128, "q_rank": width * 3 // 8 if width == 2048 else 512, "kv_rank": width // 4, "scale": 192 ** -0.5,
            "rot": {"base": 10000.0, "dims": 64}}
    ssm = {"heads": width // 32, "vdim": 64, "state": 128, "groups": width // 256, "norm_groups": width // 256, "conv": 4}
    moe = {"kind": "moe", "expert": {"ff": width * 11 // 16}, "router": {"experts": 16, "top": 4, "groups": {"count": 4, "keep": 2}}}
    layers = []
    for i in range(6):
        mixer = {**attn, **({"kv_from": 0} if i == 3 else {})}
        layers.append({"type": "latent_attention", "mixer": mixer, "mlp": {"kind": "dense", "ff": ff} if i == 0 else moe} if i % 3 == 0 else
                      {"type": "mamba2", "mixer": ssm, "mlp": moe})
    return {"architecture": "Tanolorn", "vocab": VOCAB, "width": width, "norm": {"eps": EPS}, "token_side": {"dim": width // 8}, "layers": layers}


def _shapes(design, c):
    out = {}
    if design == "llama":
        w, ff, kv = c["hidden_size"], c["intermediate_size"], c["hidden_size"] // c["num_attention_heads"] * c["num_key_value_heads"]
        out["model.embed_tokens.weight"], out["model.norm.weight"] = (VOCAB, w), (w,)
        for i in range(c["num_hidden_layers"]):
            p = f"model.layers.{i}."
            out.update({p + "input_layernorm.weight": (w,), p + "post_attention_layernorm.weight": (w,), p + "mlp.gate_proj.weight": (ff, w), p + "mlp.up_proj.weight": (ff, w),
                        p + "mlp.down_proj.weight": (w, ff), p + "self_attn.q_proj.weight": (w, w), p + "self_attn.k_proj.weight": (kv, w), p + "self_attn.v_proj.weight": (kv, w),
                        p + "self_attn.o_proj.weight": (w, w)})
        return out
    w = c["width"]
    out["embed"], out["head"], out["final.norm"] = (VOCAB, w), (VOCAB, w), (w,)
    if design == "tanolorn":
        side = c["token_side"]["dim"]
        out["side.embed"] = (VOCAB, side * len(c["layers"]))
    for i, layer in enumerate(c["layers"]):
        p, m, f = f"l{i}.", layer["mixer"], layer["mlp"]
        H = m["heads"]
        out.update({p + "norm1": (w,), p + "norm2": (w,)})
        if design == "tugelorn":
            G, d, vd = m["kv_heads"], m["dim"], m["vdim"]
            out.update({p + "norm1b": (w,), p + "norm2b": (w,), p + "mix.q": ((G if layer["type"] == "channel_delta" else H) * d, w), p + "mix.k": (G * d, w),
                        p + "mix.o": (w, H * vd), p + "mlp.gate": (f["ff"], w), p + "mlp.up": (f["ff"], w), p + "mlp.down": (w, f["ff"])})
            if layer["type"] == "channel_delta":
                out.update({p + "mix.v": (H * vd, w), p + "mix.q.conv": (G * d, m["conv"]), p + "mix.k.conv": (G * d, m["conv"]), p + "mix.v.conv": (H * vd, m["conv"]), p + "mix.b": (H, w),
                            p + "mix.A_log": (H,), p + "mix.norm": (vd,), p + "mix.a1": (d, w), p + "mix.a2": (H * d, d), p + "mix.dt_bias": (H * d,), p + "mix.g1": (vd, w),
                            p + "mix.g2": (H * vd, vd)})
            else:
                out[p + "mix.v"] = (G * vd, w)
                if layer["type"] == "attention_2":
                    out.update({p + "mix.q.b": (H * d,), p + "mix.k.b": (G * d,), p + "mix.v.b": (G * vd,)})
            continue
        if layer["type"] == "latent_attention":
            out.update({p + "mix.dq": (m["q_rank"], w), p + "mix.dq.norm": (m["q_rank"],), p + "mix.uq": (H * (m["dim"] + m["rot_dim"]), m["q_rank"]),
                        p + "mix.uk": (H * m["dim"], m["kv_rank"]), p + "mix.uv": (H * m["vdim"], m["kv_rank"]), p + "mix.o": (w, H * m["vdim"])})
            if "kv_from" not in m:
                out.update({p + "mix.dkv": (m["kv_rank"] + m["rot_dim"], w), p + "mix.dkv.norm": (m["kv_rank"],)})
        else:
            inner, ch = H * m["vdim"], H * m["vdim"] + 2 * m["groups"] * m["state"]
            out.update({p + "mix.in": (inner + ch + H, w), p + "mix.conv": (ch, m["conv"]), p + "mix.conv.b": (ch,), p + "mix.dt_bias": (H,), p + "mix.A_log": (H,), p + "mix.D": (H,),
                        p + "mix.norm": (inner,), p + "mix.o": (w, inner)})
        if f["kind"] == "dense":
            out.update({p + "mlp.gate": (f["ff"], w), p + "mlp.gate.b": (f["ff"],), p + "mlp.up": (f["ff"], w), p + "mlp.up.b": (f["ff"],), p + "mlp.down": (w, f["ff"]), p + "mlp.down.b": (w,)})
        else:
            n, e = f["router"]["experts"], f["expert"]["ff"]
            out.update({p + "mlp.router": (n, w), p + "mlp.correction": (n,)})
            for j in range(n):
                out.update({p + f"mlp.e{j}.gate": (e, w), p + f"mlp.e{j}.up": (e, w), p + f"mlp.e{j}.down": (w, e)})
        out.update({p + "side.gate": (side, w), p + "side.proj": (w, side), p + "side.norm": (w,)})
    return out


def _weights(design, c):
    """(name, bf16 tensor) one by one, the same ones every time.  Scales as in the tests' models: activations keep their size from layer
    to layer, decays run from little to much, the router spreads rows over its experts."""
    gen = torch.Generator(device="cuda").manual_seed(9)
    for name, shape in _shapes(design, c).items():
        x, tail = torch.randn(shape, device="cuda", generator=gen), name.split(".")[-1]
        if design == "llama":
            x = 1 + 0.02 * x if len(shape) == 1 else 0.3 * x if "embed" in name else x / math.sqrt(shape[-1])
        elif design == "tanolorn" and (tail in ("norm1", "norm2") or name == "final.norm"):
            x = 0.1 * x  # stored around zero
        elif "norm" in tail or tail == "D":
            x = 1 + 0.1 * x
        elif tail == "A_log":
            x = 0.7 * x - 1
        elif tail == "dt_bias":
            x = x - 1.5
        elif tail == "conv":
            x = 0.5 * x
        elif tail == "correction":
            x = 0.1 * x
        elif len(shape) == 1:
            x = 0.2 * x
        elif name not in ("embed", "side.embed"):
            x = x / math.sqrt(shape[-1])
        yield name, x.bfloat16()


# ---- what a program keeps --------------------------------------------------------------------------------------------------------
_kept = {}


def _device():
    if "device" not in _kept:
        _kept["device"] = ug_amd.hip_device(0)
        _kept["device"].set_zero_fill(False)  # as bin/generate and bin/trace_run set it
    return _kept["device"]


def _model(case):
    """A program loads its model once, from a folder, and then answers many prompts; the last two stay."""
    key = case["design"], case["width"], case["dtype"]
    models = _kept.setdefault("models", {})
    if key not in models:
        if len(models) > 1:
            del models[next(iter(models))]
        config, folder = _config(*key[:2]), tempfile.mkdtemp()
        try:
            with open(os.path.join(folder, "config.json"), "w") as f:
                json.dump(config, f)
            st_writer.write_safetensors(os.path.join(folder, "model.safetensors"),
                                        [(n, "BF16", tuple(x.shape), x.view(torch.int16).cpu().numpy().view(np.uint16)) for n, x in _weights(key[0], config)])
            models[key] = ug_amd.Decoder.load(_device(), folder, bf16=key[2] == "bf16")
        finally:
            shutil.rmtree(folder)
    return models[key]


class _Memory:
    """Device memory of the framework, as torch takes it in."""

    def __init__(self, ptr, shape, typestr):
        self.__cuda_array_interface__ = {"shape": shape, "typestr": typestr, "data": (ptr, False), "version": 3}


def _view(slice_, shape, dtype):
    ptr = ug_amd.ughip_lib().ughip_slice_ptr(ctypes.c_void_p(slice_.raw()))
    return torch.as_tensor(_Memory(ptr, shape, "<f4" if dtype == "f32" else "<i2"), device="cuda").view(TORCH[dtype])


def _view_of_buffer(lb, shape):
    """The realised storage of a lazy buffer, through a custom op that is handed its slice."""
    seen = []
    probe = LB.custom(lambda slices: seen.append(_view(slices[0], shape, "f32")), [lb], (1,), ug_amd.F32, _device())
    Schedule.create_one(probe).compile().run()
    return seen[0]


# ---- inputs ----------------------------------------------------------------------------------------------------------------------
def _normal(seed, i, shape, dtype="f32"):
    return torch.randn(shape, device="cuda", generator=torch.Generator(device="cuda").manual_seed(seed * 16 + i)).to(TORCH[dtype])


def _inputs(case, seed):
    if case["kind"] == "rows":
        x = _normal(seed, 0, (case["rows"], case["cols"]))
        return (3 * x,) if case["op"] == "softmax" else (x, 1 + 0.1 * _normal(seed, 1, (case["cols"],)))
    if case["kind"] == "reduce":
        gen = torch.Generator(device="cuda").manual_seed(seed)
        return tuple(torch.rand(case["n"], device="cuda", generator=gen) for _ in range(2))
    if case["kind"] == "product":
        b, m, n, k = (case[d] for d in "bmnk")
        return _normal(seed, 0, (b, m, k), case["dtype"]), _normal(seed, 1, (b, n, k) if case["nt"] else (b, k, n), case["dtype"])
    return np.random.default_rng(seed).integers(0, VOCAB, case["prompt"] + case.get("steps", 0), dtype=np.int32)


def prepare(case, seed):
    dev, x = _device(), _inputs(case, seed)
    if case["kind"] in ("rows", "reduce"):
        args = [LB.copy(t.cpu().numpy(), tuple(t.shape), dev) for t in x]
        if case["kind"] == "reduce":
            out, shape = fused_reduce_graph(*args, dev), (1,)
        else:
            out, shape = ug_amd.llama.softmax(args[0]) if case["op"] == "softmax" else ug_amd.llama.rms_norm(*args, EPS), tuple(x[0].shape)
        compiled = Schedule.create_one(out).compile()
        compiled.run()
        return {"compiled": compiled, "out": out, "view": _view_of_buffer(out, shape)}
    if case["kind"] == "product":
        b, m, n, k = (case[d] for d in "bmnk")
        slices = [dev.allocate_uninit(UG[case["dtype"]], size) for size in (b * m * n, b * m * k, b * n * k)]
        for s, t in zip(slices[1:], x):
            _view(s, tuple(t.shape), case["dtype"]).copy_(t)
        torch.cuda.synchronize()
        rhs = ([b, k, n], [n * k, 1, k] if case["nt"] else [n * k, n, 1], 0)
        return {"args": (*slices, (b, m, n, k), ([b, m, k], [m * k, k, 1], 0), rhs), "view": _view(slices[0], (b, m, n), case["dtype"])}
    return {"model": _model(case), "prompt": x[: case["prompt"]], "reply": x[case["prompt"] :]}


def run(state):
    if "compiled" in state:
        state["compiled"].run()
        return state["view"]
    if "args" in state:
        _device().matmul(*state["args"])
        return state["view"]
    model, prompt, reply = state["model"], state["prompt"], state["reply"]
    if not len(reply):
        return model.step(model.new_state(len(prompt)), prompt, want=[len(prompt) - 1])
    # the reply's ids are given (a known text is scored), so that a tie cannot lead two runs apart
    ids, stats = model.generate(prompt, len(reply), forced=reply)
    return {"ids": ids, "top": stats["top1"], "margin": stats["margins"]}


# ---- what a pass cannot do without -----------------------------------------------------------------------------------------------
def work(case):
    if case["kind"] == "rows":
        n = case["rows"] * case["cols"]
        return {"bytes": 8 * n, "flops": 5 * n}
    if case["kind"] == "reduce":
        return {"bytes": 8 * case["n"], "flops": 4 * case["n"]}
    if case["kind"] == "product":
        b, m, n, k = (case[d] for d in "bmnk")
        return {"bytes": b * (m * n + m * k + n * k) * (4 if case["dtype"] == "f32" else 2), "flops": 2 * b * m * n * k}
    # weights: a prompt reads all of them once, a single position those that act on it; an embedding is read by row.  Every position's
    # row meets the matrices that act on it, the head meets the rows whose logits are asked for.
    config, per = _config(case["design"], case["width"]), 2 if case["dtype"] == "bf16" else 4
    held = acting = 0
    for name, shape in _shapes(case["design"], config).items():
        if "embed" in name or name == "head" or len(shape) == 1:
            continue
        held += shape[0] * shape[1]
        acting += shape[0] * shape[1] // (4 if ".mlp.e" in name else 1)
    head, t, steps = VOCAB * case["width"], case["prompt"], case.get("steps", 0)
    pairs, row = t * t // 2 + steps * (t + steps // 2), 0  # positions that meet, and what they exchange
    for layer in config.get("layers", [None] * 6):
        m = layer["mixer"] if layer else {}
        if not layer or layer["type"] in ("attention", "attention_2", "latent_attention"):
            row += 4 * case["width"] if layer is None or "rot_dim" not in m else 2 * m["heads"] * (m["dim"] + m["rot_dim"] + m["vdim"])
        else:
            acting += 3 * m["heads"] * m["vdim"] * m.get("state", m.get("dim"))  # the recurrence's state, decayed, written and read
    return {"bytes": per * (held + head + steps * (acting + head)), "flops": 2 * acting * (t + steps) + 2 * head * (1 + steps) + row * pairs}


def tolerance(case):
    """About four times the error measured against `exact` over the ranges of `draw`."""
    if case["kind"] in ("rows", "reduce"):
        return {"rel": 2e-6}
    if case["kind"] == "product":
        return {"rel": {"f32": 5e-6, "f16": 1e-3, "bf16": 7e-3}[case["dtype"]]}
    if case["dtype"] == "f32" or case["design"] == "llama":  # the llama's rows meet bf16 matrices as three bf16 terms, 24 bits in all
        return {"rel": 5e-5, "max": 5e-3, "differ": 0.01}
    # rows rounded to bf16 in front of products; with experts a rounding may also turn a choice
    return {"rel": 3e-2 if case["design"] == "tanolorn" else 1.5e-2, "max": 0.5, "differ": 0.01}


# ---- the same in 64 bits ---------------------------------------------------------------------------------------------------------
def _rms(x, eps=EPS):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)


def _silu(x):
    return x * torch.sigmoid(x)


def _rotate(x, base, dims, factor=1.0, pairs=False, single=False):
    """x [t, heads, d]: the first `dims` elements by the position's angles, halves (or neighbours) in pairs.  single: frequencies
    rounded to 32 bits, as the llama defines them."""
    if single:
        freq = torch.tensor([float(np.float32(1) / np.float32(base) ** (np.float32(i) / np.float32(dims))) for i in range(0, dims, 2)], dtype=torch.float64, device=x.device)
    else:
        freq = base ** (-torch.arange(0, dims, 2, dtype=torch.float64, device=x.device) / dims) / factor
    a = torch.arange(len(x), dtype=torch.float64, device=x.device)[:, None] * freq
    c, s, out = a.cos()[:, None], a.sin()[:, None], x.clone()
    u, v = (slice(0, dims, 2), slice(1, dims, 2)) if pairs else (slice(0, dims // 2), slice(dims // 2, dims))
    out[..., u], out[..., v] = x[..., u] * c - x[..., v] * s, x[..., v] * c + x[..., u] * s
    return out


def _attend(q, k, v, scale, window=None):
    """q [t, H, d], k and v [t, G, ..]: causal, grouped heads, optionally the last `window` positions only -> [t, H * vd]."""
    t, H, per = len(q), q.shape[1], q.shape[1] // k.shape[1]
    i = torch.arange(t, device=q.device)
    hidden = (i[None, :] > i[:, None]) | ((i[:, None] - i[None, :] >= window) if window else False)
    out = []
    for h in range(H):
        s = (q[:, h].contiguous() @ k[:, h // per].contiguous().T) * scale
        out.append(torch.softmax(s.masked_fill(hidden, -math.inf), -1) @ v[:, h // per].contiguous())
    return torch.cat(out, 1)


def _conv(x, taps):
    n = taps.shape[1]
    pad = torch.cat([x.new_zeros(n - 1, x.shape[1]), x])
    return sum(pad[j : j + len(x)] * taps[:, j] for j in range(n))


def _llama(c, w, tokens):
    t, H, G = len(tokens), c["num_attention_heads"], c["num_key_value_heads"]
    d, x = c["hidden_size"] // H, w["model.embed_tokens.weight"][tokens]
    for i in range(c["num_hidden_layers"]):
        g = lambda n: w[f"model.layers.{i}.{n}.weight"]  # noqa: B023,E731
        h = _rms(x) * g("input_layernorm")
        q, k, v = ((h @ g(f"self_attn.{n}_proj").T).reshape(t, -1, d) for n in "qkv")
        q, k = (_rotate(y, 10000.0, d, single=True) for y in (q, k))
        x = x + _attend(q, k, v, d ** -0.5) @ g("self_attn.o_proj").T
        h = _rms(x) * g("post_attention_layernorm")
        x = x + (_silu(h @ g("mlp.gate_proj").T) * (h @ g("mlp.up_proj").T)) @ g("mlp.down_proj").T
    return _rms(x) * w["model.norm.weight"], w["model.embed_tokens.weight"]


def _latent(x, w, m, latents, i):
    t, H, d, r = len(x), m["heads"], m["dim"], m["rot_dim"]
    if "kv_from" in m:
        c, k_rot = latents[m["kv_from"]]
    else:
        kv = x @ w["dkv"].T
        c, k_rot = latents[i] = _rms(kv[:, : m["kv_rank"]]) * w["dkv.norm"], _rotate(kv[:, None, m["kv_rank"] :], m["rot"]["base"], r)
    q = ((_rms(x @ w["dq"].T) * w["dq.norm"]) @ w["uq"].T).reshape(t, H, d + r)
    q = torch.cat([q[..., :d], _rotate(q[..., d:], m["rot"]["base"], r)], -1)
    k = torch.cat([(c @ w["uk"].T).reshape(t, H, d), k_rot.expand(t, H, r)], -1)
    return _attend(q, k, (c @ w["uv"].T).reshape(t, H, m["vdim"]), m["scale"]) @ w["o"].T


def _mamba2(x, w, m):
    t, H, vd, N, G = len(x), m["heads"], m["vdim"], m["state"], m["groups"]
    z, xbc, dt = (x @ w["in"].T).split([H * vd, H * vd + 2 * G * N, H], 1)
    u, B, C = _silu(_conv(xbc, w["conv"]) + w["conv.b"]).split([H * vd, G * N, G * N], 1)
    u, B, C = u.reshape(t, H, vd), *(y.reshape(t, G, N).repeat_interleave(H // G, 1) for y in (B, C))
    dt = torch.logaddexp(dt + w["dt_bias"], torch.zeros_like(dt))
    decay, S, y = torch.exp(-torch.exp(w["A_log"]) * dt), x.new_zeros(H, N, vd), []
    for i in range(t):
        S = decay[i, :, None, None] * S + (dt[i, :, None] * B[i])[:, :, None] * u[i, :, None, :]
        y.append((C[i, :, :, None] * S).sum(1))
    y = ((torch.stack(y) + w["D"][:, None] * u).reshape(t, -1) * _silu(z)).reshape(t, m["norm_groups"], -1)
    return (_rms(y).reshape(t, -1) * w["norm"]) @ w["o"].T


def _experts(x, w, f):
    r, t = f["router"], len(x)
    s = torch.sigmoid(x @ w["router"].T)
    choice = s + w["correction"]
    best = choice.reshape(t, r["groups"]["count"], -1).topk(2, -1).values.sum(-1).topk(r["groups"]["keep"], -1).indices
    shut = torch.ones(t, r["groups"]["count"], dtype=torch.bool, device=x.device).scatter(1, best, False).repeat_interleave(r["experts"] // r["groups"]["count"], 1)
    acts = torch.zeros_like(shut).scatter(1, choice.masked_fill(shut, -math.inf).topk(r["top"], -1).indices, True)
    out = torch.zeros_like(x)
    for e in range(r["experts"]):
        at = acts[:, e].nonzero()[:, 0]
        h = x[at]
        out[at] += s[at, e, None] * ((_silu(h @ w[f"e{e}.gate"].T) * (h @ w[f"e{e}.up"].T)) @ w[f"e{e}.down"].T)
    return out


def _under(w, prefix):
    return {k[len(prefix) :]: v for k, v in w.items() if k.startswith(prefix)}


def _tanolorn(c, w, tokens):
    x, side, latents = w["embed"][tokens], c["token_side"]["dim"], {}
    for i, layer in enumerate(c["layers"]):
        p, f = f"l{i}.", layer["mlp"]
        mix, ff = _under(w, p + "mix."), _under(w, p + "mlp.")
        y = _latent(x, mix, layer["mixer"], latents, i) if layer["type"] == "latent_attention" else _mamba2(x, mix, layer["mixer"])
        x = x + _rms(y) * (1 + w[p + "norm1"])
        y = _experts(x, ff, f) if f["kind"] == "moe" else (_silu(x @ ff["gate"].T + ff["gate.b"]) * (x @ ff["up"].T + ff["up.b"])) @ ff["down"].T + ff["down.b"]
        x = x + _rms(y) * (1 + w[p + "norm2"])
        gate = torch.nn.functional.gelu(x @ w[p + "side.gate"].T, approximate="tanh")
        x = x + _rms((gate * w["side.embed"][tokens, i * side : (i + 1) * side]) @ w[p + "side.proj"].T) * w[p + "side.norm"]
    return _rms(x) * (1 + w["final.norm"]), w["head"]


def _delta(h, w, m):
    t, H, G, d, vd = len(h), m["heads"], m["kv_heads"], m["dim"], m["vdim"]
    q, k, v = (_silu(_conv(h @ w[n].T, w[n + ".conv"])) for n in "qkv")
    unit = lambda y: y * torch.rsqrt((y * y).sum(-1, keepdim=True) + 1e-6)  # noqa: E731
    q, k, v = unit(q.reshape(t, G, d)) * d ** -0.5, unit(k.reshape(t, G, d)), v.reshape(t, H, vd)
    q, k = (y.repeat_interleave(H // G, 1) for y in (q, k))
    step = h @ w["a1"].T @ w["a2"].T + w["dt_bias"]
    decay = torch.exp(-torch.exp(w["A_log"])[:, None] * torch.logaddexp(step, torch.zeros_like(step)).reshape(t, H, d))
    beta, S, out = torch.sigmoid(h @ w["b"].T), h.new_zeros(H, d, vd), []
    for i in range(t):
        S = S * decay[i, :, :, None]
        u = beta[i, :, None] * (v[i] - (S * k[i, :, :, None]).sum(1))
        S = S + k[i, :, :, None] * u[:, None]
        out.append((S * q[i, :, :, None]).sum(1))
    o = _rms(torch.stack(out)) * w["norm"] * torch.sigmoid(h @ w["g1"].T @ w["g2"].T).reshape(t, H, vd)
    return o.reshape(t, -1) @ w["o"].T


def _grouped(h, w, m, kind):
    t = len(h)
    q, k, v = ((h @ w[n].T + (w[n + ".b"] if kind == "attention_2" else 0)).reshape(t, -1, m["vdim" if n == "v" else "dim"]) for n in "qkv")
    if kind == "attention":
        q, k = (_rotate(y, m["rot"]["base"], m["rot"]["dims"], m["rot"]["scaling"]["factor"], pairs=True) for y in (q, k))
        return _attend(q, k, v, m["scale"], m["mask"]["size"]) @ w["o"].T
    at = torch.arange(t, dtype=torch.float64, device=h.device)
    q = q * (1 + m["q_temp"]["coef"] * torch.log(torch.floor((at + 1) / m["q_temp"]["every"]) + 1))[:, None, None]
    return _attend(q, k, v, m["scale"]) @ w["o"].T


def _tugelorn(c, w, tokens):
    x, r = w["embed"][tokens], c["residual_mult"]
    norm = lambda y, n: _rms(y) * w[n]  # noqa: E731
    for i, layer in enumerate(c["layers"]):
        p, mix = f"l{i}.", _under(w, f"l{i}.mix.")
        h = norm(x, p + "norm1")
        y = _delta(h, mix, layer["mixer"]) if layer["type"] == "channel_delta" else _grouped(h, mix, layer["mixer"], layer["type"])
        x = x + r * norm(y, p + "norm1b")
        h, cut = norm(x, p + "norm2"), layer["mlp"]["limit"]
        g, u = (h @ w[p + "mlp.gate"].T).clamp(max=cut), (h @ w[p + "mlp.up"].T).clamp(-cut, cut)
        x = x + r * norm((g * torch.sigmoid(1.702 * g) * (u + 1)) @ w[p + "mlp.down"].T, p + "norm2b")
    return norm(x, "final.norm"), w["head"]


def exact(case, seed):
    x = _inputs(case, seed)
    if case["kind"] == "rows":
        x = [t.double() for t in x]
        return torch.softmax(x[0], -1) if case["op"] == "softmax" else _rms(x[0]) * x[1]
    if case["kind"] == "reduce":
        a, b = (t.double() for t in x)
        return (a * b + 0.5 * a).sum().reshape(1)
    if case["kind"] == "product":
        a, b = (t.double() for t in x)
        return torch.stack([p @ (q.T if case["nt"] else q) for p, q in zip(a, b)])
    design, config = case["design"], _config(case["design"], case["width"])
    w = {n: t.double() for n, t in _weights(design, config)}
    rows, head = {"llama": _llama, "tanolorn": _tanolorn, "tugelorn": _tugelorn}[design](config, w, torch.from_numpy(x).long().cuda())
    logits = rows[case["prompt"] - 1 :] @ head.T
    if case["kind"] == "prompt":
        return logits
    two = logits.topk(2, -1)
    return {"ids": two.indices[:, 0], "top": two.values[:, 0], "margin": two.values[:, 0] - two.values[:, 1]}
