"""Workloads of the library, each one pass through the entry points of include/kx.h as a program that uses it calls them.

Three kinds of case:
  moe    : one routed-MoE layer at Kimi-K2 shape on activations in device memory (kx_moe_decode_layer, kx_moe_prefill_layer)
  mla    : latent decode attention over a cache in device memory (kx_mla_decode)
  model  : a resident model; the pass is a prompt (steps 0) or a prompt and a number of decode steps whose ids the
           program chooses (a sampler on the host, constrained decoding, replay), and the pass returns the logits it asked for.
           Designs: "kimi" (kx_model_create), "kagalorn" and "rapitar" (config.json and safetensors, kx_model_open).

Weights, activations and ids are random, made from the seed; sizes are those of bench.py's workloads, of the
default configuration and of tests/, and sizes around them.
"""
import ctypes as C
import json
import math
import os
import shutil
import struct
import tempfile

import numpy as np
import torch

from blok_amd.lib import DTYPES, KxMoeWeights, KxOpenOptions, check, default_config, kx

E, TOP, HIDDEN, INTER = 384, 8, 7168, 2048          # the routed layer of Kimi-K2 (kx_config_default)
NOPE, ROPE, VHEAD, KV_RANK, Q_RANK = 128, 64, 128, 512, 1536
SCALE = 2.827                                       # routed_scale


def listed():
    return [
        # one token of one sequence through the MoE layer: what every decoded token of an interactive session pays per layer
        {"name": "moe 1", "kind": "moe", "path": "decode", "tokens": 1},
        # a served batch of decoding sequences through the same layer, with the kernels that the decoder stack asks for there
        {"name": "moe 24", "kind": "moe", "path": "batch", "tokens": 24},
        # a full prefill step through the layer, routing skewed as trained routers' is
        {"name": "moe prompt 2048", "kind": "moe", "path": "prompt", "tokens": 2048},
        # latent attention of a batch of long sequences
        {"name": "mla 16 x 32768", "kind": "mla", "batch": 16, "context": 32768},
        # interactive decoding on the Kimi-K2 stack (cut to a dense and two MoE layers), one sequence, the bit-reproducible path
        {"name": "kimi reply", "kind": "model", "design": "kimi", "dtype": "bfloat16", "width": 7168, "heads": 64, "ff": 18432, "layers": 3,
         "moe_layers": 2, "vocab": 32768, "batch": 1, "prompt": 600, "steps": 16},
        # a long prompt through dense layers of that stack in prefill steps of 2048 positions
        {"name": "kimi prompt", "kind": "model", "design": "kimi", "dtype": "bfloat16", "width": 7168, "heads": 64, "ff": 18432, "layers": 2,
         "moe_layers": 0, "vocab": 32768, "batch": 1, "prompt": 3000, "steps": 0},
        # a served batch decoding on the same layers, contexts of ordinary length
        {"name": "kimi batch", "kind": "model", "design": "kimi", "dtype": "bfloat16", "width": 7168, "heads": 64, "ff": 18432, "layers": 2,
         "moe_layers": 0, "vocab": 32768, "batch": 12, "prompt": 1500, "steps": 8},
        # a long prompt for the Kagalorn design at the smallest width of the benchmark
        {"name": "kagalorn prompt", "kind": "model", "design": "kagalorn", "dtype": "bfloat16", "width": 2048, "heads": 16, "kv_heads": 4, "ff": 8192,
         "layers": 4, "vocab": 16384, "batch": 1, "prompt": 4096, "steps": 0},
        # an interactive answer from it
        {"name": "kagalorn reply", "kind": "model", "design": "kagalorn", "dtype": "bfloat16", "width": 2048, "heads": 16, "kv_heads": 4, "ff": 8192,
         "layers": 4, "vocab": 16384, "batch": 1, "prompt": 300, "steps": 48},
        # several prompts of odd length together through the Rapitar design (state space, time mixing, latent attention, experts)
        {"name": "rapitar prompts", "kind": "model", "design": "rapitar", "dtype": "bfloat16", "width": 2048, "heads": 16, "kv_heads": 4, "ff": 8192,
         "layers": 4, "vocab": 16384, "batch": 3, "prompt": 701, "steps": 0},
        # a served batch decoding on it
        {"name": "rapitar batch", "kind": "model", "design": "rapitar", "dtype": "bfloat16", "width": 2048, "heads": 16, "kv_heads": 4, "ff": 8192,
         "layers": 4, "vocab": 16384, "batch": 8, "prompt": 60, "steps": 24},
        # the 32-bit format, as it is used to check a model's bf16 results
        {"name": "kagalorn prompt f32", "kind": "model", "design": "kagalorn", "dtype": "float32", "width": 1024, "heads": 8, "kv_heads": 2, "ff": 4096,
         "layers": 4, "vocab": 8192, "batch": 1, "prompt": 777, "steps": 0},
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, spread evenly over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["moe", "mla", "kimi", "kimi", "hybrid", "hybrid", "hybrid", "hybrid"])
    if kind == "moe":
        path = rng.choice(["decode", "batch", "prompt"])
        tokens = _log(rng, *{"decode": (2, 12), "batch": (5, 64), "prompt": (33, 2047)}[path])
        return {"kind": "moe", "path": path, "tokens": tokens}
    if kind == "mla":
        batch = _log(rng, 1, 32)
        return {"kind": "mla", "batch": batch, "context": _log(rng, 100, min(131072, 500000 // batch))}
    if kind == "kimi":
        heads, width, ff = rng.choice([(16, 2048, 8192), (32, 4096, 12288), (64, 7168, 18432)])
        c = {"kind": "model", "design": "kimi", "dtype": "bfloat16", "width": width, "heads": heads, "ff": ff, "layers": 2, "moe_layers": 0, "vocab": 16384}
        if rng.random() < 0.5:
            batch = _log(rng, 1, 4)
            return {**c, "batch": batch, "prompt": _log(rng, 40, 2500 // batch), "steps": 0}
        batch = _log(rng, 1, 32)
        return {**c, "batch": batch, "prompt": _log(rng, 40, min(2000, 12000 // batch)), "steps": rng.randint(3, 8)}
    width, heads = rng.choice([(1024, 8), (1536, 12), (2048, 16)])
    dtype = rng.choice(["bfloat16", "bfloat16", "bfloat16", "float32"])
    design = rng.choice(["kagalorn", "rapitar"])
    if dtype == "float32":
        width, heads = 1024, 8
    kv = rng.choice([k for k in (2, 4, 8) if heads % k == 0])
    c = {"kind": "model", "design": design, "dtype": dtype, "width": width, "heads": heads, "kv_heads": kv,
         "ff": rng.choice([2, 3, 4]) * width + 8 * rng.randint(0, 7), "layers": 4, "vocab": 1024 * rng.randint(4, 16) + rng.randint(0, 9)}
    if rng.random() < 0.5:
        batch = _log(rng, 1, 4)
        return {**c, "batch": batch, "prompt": _log(rng, 20, (800 if dtype == "float32" else 4000) // batch), "steps": 0}
    if dtype == "float32":
        batch = _log(rng, 1, 16)
        return {**c, "batch": batch, "prompt": _log(rng, 10, 800 // batch), "steps": rng.randint(4, 12)}
    batch = _log(rng, 1, 32)
    return {**c, "batch": batch, "prompt": _log(rng, 10, min(1000, 4000 // batch)), "steps": rng.randint(8, 32)}


# ---- inputs -------------------------------------------------------------------------------------------------------
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _bf16(g, shape, sigma, magnitude=False):
    x = torch.randn(shape, generator=g, device="cuda", dtype=torch.bfloat16).mul_(sigma)
    return x.abs_() if magnitude else x


class _Held:
    """A handle of the library that goes back when the state does."""

    def __init__(self, handle, destroy):
        self.h, self._destroy = handle, destroy

    def __del__(self):
        try:
            self._destroy(self.h)
        except Exception:
            pass


def _moe_inputs(case, seed):
    g, t = _generator(seed), case["tokens"]
    words = lambda n, k: torch.randint(-2 ** 31, 2 ** 31 - 1, (E, n, k // 8), generator=g, device="cuda", dtype=torch.int32)
    scale = lambda n, k: _bf16(g, (E, n, k // 32), 0.02, magnitude=True)
    w = {"router_gate": _bf16(g, (E, HIDDEN), HIDDEN ** -0.5)}
    if case["path"] == "prompt":   # a few experts take most tokens
        rank = torch.randperm(E, generator=g, device="cuda").float() + 1
        w["router_bias"] = -0.1 * rank.log()
    else:
        w["router_bias"] = torch.randn(E, generator=g, device="cuda") * 0.01
    for name, n, k in (("gate", INTER, HIDDEN), ("up", INTER, HIDDEN), ("down", HIDDEN, INTER)):
        w[name + "_packed"], w[name + "_scale"] = words(n, k), scale(n, k)
    w["shared_gate"], w["shared_up"], w["shared_down"] = _bf16(g, (INTER, HIDDEN), 0.02), _bf16(g, (INTER, HIDDEN), 0.02), _bf16(g, (HIDDEN, INTER), 0.02)
    return w, _bf16(g, (t, HIDDEN), 1.0), _bf16(g, (t, HIDDEN), 1.0)


def _prepare_moe(case, seed):
    w, n, x = _moe_inputs(case, seed)
    cfg, mw, ws = default_config(), KxMoeWeights(), C.c_void_p()
    for name, v in w.items():
        setattr(mw, "d_" + name, v.data_ptr())
    check(kx().kx_moe_workspace_create(C.byref(cfg), case["tokens"], C.byref(ws)))
    return {"case": case, "w": w, "mw": mw, "cfg": cfg, "n": n, "x": x, "ws": _Held(ws, kx().kx_moe_workspace_destroy)}


def _run_moe(s):
    case = s["case"]
    call = kx().kx_moe_prefill_layer if case["path"] == "prompt" else kx().kx_moe_decode_layer
    flags = 0x600 if case["path"] == "batch" else 0
    check(call(C.byref(s["cfg"]), C.byref(s["mw"]), s["ws"].h, s["n"].data_ptr(), s["x"].data_ptr(), case["tokens"], flags, None))
    return s["x"]                  # the residual stream, updated in place


def _mla_inputs(case, seed):
    g = _generator(seed)
    cache = _bf16(g, (case["batch"], case["context"], KV_RANK + ROPE), 1.0)
    q = _bf16(g, (case["batch"], 64, KV_RANK + ROPE), 0.6).float()
    return cache, q


def _prepare_mla(case, seed):
    cache, q = _mla_inputs(case, seed)
    cfg, size = default_config(), C.c_size_t()
    check(kx().kx_mla_workspace_bytes(C.byref(cfg), case["batch"], case["context"], C.byref(size)))
    return {"case": case, "cfg": cfg, "cache": cache, "q": q, "work": torch.empty(size.value, dtype=torch.uint8, device="cuda"),
            "out": torch.empty((case["batch"], 64, KV_RANK), dtype=torch.bfloat16, device="cuda")}


def _run_mla(s):
    case = s["case"]
    check(kx().kx_mla_decode(C.byref(s["cfg"]), s["cache"].data_ptr(), case["context"] * (KV_RANK + ROPE), s["q"].data_ptr(),
                             s["work"].data_ptr(), s["out"].data_ptr(), case["batch"], case["context"], 0, None))
    return s["out"]


def _ids(case, seed):
    """[batch][prompt + steps]"""
    return np.random.default_rng(seed).integers(0, case["vocab"], (case["batch"], case["prompt"] + case["steps"])).astype(np.uint32)


def _kimi_config(case, seed):
    c = default_config()
    c.n_layers, c.first_dense = case["layers"], case["layers"] - case["moe_layers"]
    c.hidden, c.heads, c.dense_inter, c.vocab = case["width"], case["heads"], case["ff"], case["vocab"]
    c.max_batch, c.max_context, c.seed = case["batch"], case["prompt"] + case["steps"], seed
    return c


def _hybrid_config(case):
    w, heads, kv, ff = case["width"], case["heads"], case["kv_heads"], case["ff"]
    if case["design"] == "kagalorn":
        mlp = {"kind": "dense", "ff": ff, "limit": 7.0}
        attn = {"type": "attention", "mlp": mlp, "mixer": {"heads": heads, "kv_heads": kv, "dim": 128, "vdim": 128, "scale": 128 ** -0.5,
                                                           "mask": {"size": 1024, "pool": 16}}}
        delta = {"type": "delta", "mlp": mlp, "mixer": {"heads": heads, "kv_heads": heads // 2, "dim": 128, "vdim": 128, "conv": 4}}
        layers, more = [attn, delta] * 2, {"architecture": "Kagalorn", "streams": 2, "norm": {"eps": 1e-5, "groups": 2}}
    else:
        dense, moe = {"kind": "dense", "ff": ff}, {"kind": "moe", "expert": {"ff": ff // 8}, "router": {"experts": 64, "top": 8}}
        ssd = {"heads": 2 * w // 64, "vdim": 64, "state": 128, "groups": kv, "norm_groups": kv, "conv": 4}
        latent = {"heads": heads, "dim": 128, "rot_dim": 64, "vdim": 128, "q_rank": 768, "kv_rank": 512, "scale": 192 ** -0.5, "rot": {"dims": 64, "base": 10000.0}}
        layers = [{"type": t, "mixer": m, "mlp": f} for t, m, f in
                  (("mamba2", ssd, dense), ("wkv", {"heads": w // 64, "dim": 64}, moe), ("latent_attention", latent, dense), ("mamba2", ssd, moe))]
        more = {"architecture": "Rapitar", "norm": {"eps": 1e-5}}
    return {"vocab": case["vocab"], "width": w, "layers": layers[:case["layers"]], **more}


def _hybrid_shapes(cfg):
    w = cfg["width"]
    out = {"embed": (cfg["vocab"], w), "final.norm": (w,), "head": (cfg["vocab"], w)}
    for i, layer in enumerate(cfg["layers"]):
        m, mlp, h = layer["mixer"], layer["mlp"], layer["mixer"]["heads"]
        t = {"norm1": (w,)}
        if layer["type"] in ("attention", "delta"):
            k, d, v = m["kv_heads"], m["dim"], m["vdim"]
            t.update({"mix.o": (w, h * v), "mix.g": (h * v, w), "mix.k": (k * d, w)})
            if layer["type"] == "attention":
                t.update({"mix.q": (h * d, w), "mix.v": (k * v, w), "mix.q.norm": (h * d,), "mix.k.norm": (k * d,)})
            else:
                t.update({"mix.q": (k * d, w), "mix.v": (h * v, w), "mix.b": (h, w), "mix.a": (h, w), "mix.A_log": (h,), "mix.dt_bias": (h,),
                          "mix.norm": (v,), "mix.q.conv": (k * d, 4), "mix.k.conv": (k * d, 4), "mix.v.conv": (h * v, 4)})
            t.update({"norm2": (w,), "mlp.gate": (mlp["ff"], w), "mlp.up": (mlp["ff"], w), "mlp.down": (w, mlp["ff"])})
            for q in (1, 2):
                t.update({f"hc{q}.in": (cfg["streams"],), f"hc{q}.out": (cfg["streams"],), f"hc{q}.mix": (cfg["streams"],) * 2})
        else:
            if layer["type"] == "mamba2":
                inner, bc = h * m["vdim"], 2 * m["groups"] * m["state"]
                t.update({"mix.in": (2 * inner + bc + h, w), "mix.conv": (inner + bc, 4), "mix.conv.b": (inner + bc,), "mix.dt_bias": (h,),
                          "mix.A_log": (h,), "mix.D": (h,), "mix.norm": (inner,), "mix.o": (w, inner)})
            elif layer["type"] == "wkv":
                hd = h * m["dim"]
                t.update({"mix.mu." + c: (w,) for c in "rkvgw"})
                t.update({"mix." + c: (hd, w) for c in "rkvg"})
                t.update({"mix.w1": (64, w), "mix.w2": (hd, 64), "mix.w0": (hd,), "mix.u": (h, m["dim"]), "mix.norm": (hd,), "mix.o": (w, hd)})
            else:
                q, k = m["dim"] + m["rot_dim"], m["kv_rank"]
                t.update({"mix.dq": (m["q_rank"], w), "mix.dq.norm": (m["q_rank"],), "mix.uq": (h * q, m["q_rank"]), "mix.dkv": (k + m["rot_dim"], w),
                          "mix.dkv.norm": (k,), "mix.uk": (h * m["dim"], k), "mix.uv": (h * m["vdim"], k), "mix.sink": (h,),
                          "mix.g": (h * m["vdim"], w), "mix.o": (w, h * m["vdim"])})
            if mlp["kind"] == "dense":
                t.update({"mlp.up": (mlp["ff"], w), "mlp.down": (w, mlp["ff"])})
            else:
                n, f = mlp["router"]["experts"], mlp["expert"]["ff"]
                t.update({"mlp.router": (n, w), "mlp.router.b": (n,)})
                for j in range(n):
                    t.update({f"mlp.e{j}.gate": (f, w), f"mlp.e{j}.up": (f, w), f"mlp.e{j}.down": (w, f)})
        out.update({f"l{i}.{k}": v for k, v in t.items()})
    return out


def _hybrid_weights(cfg, seed):
    """bf16 tensors by name, every mechanism of a size that matters in the logits.  Routers read channels of their own that no
    layer writes to, with evenly spaced levels, so that the choice of experts has a margin as a trained router's has."""
    g, w = _generator(seed), {}
    for name, shape in _hybrid_shapes(cfg).items():
        leaf = name.split(".", 1)[-1]
        z = torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)
        if leaf.startswith("hc"):
            z = {"in": 0.5 + 0.2 * z, "out": 0.7 + 0.2 * z, "mix": 0.2 * z}[leaf[4:]]
            if leaf.endswith("mix"):
                z += torch.eye(shape[0], device="cuda")
        elif leaf.endswith("conv"):
            z *= 0.4
            z[:, -1] += 1.0
        elif leaf.endswith("A_log"):
            z = 0.8 * z - 1.0
        elif leaf.endswith(("dt_bias", "w0")):
            z = 0.5 * z - 1.5
        elif leaf in ("mix.u", "mix.sink"):
            z *= 0.8
        elif leaf.startswith("mix.mu"):
            z = 0.5 + 0.4 * z
        elif leaf in ("mix.conv.b", "mlp.router.b"):
            z *= 0.02
        elif len(shape) == 1:
            z = 0.2 * z + (0.0 if cfg["architecture"] == "Rapitar" and leaf in ("norm1", "norm") else 1.0)
        elif name != "embed":
            z *= shape[1] ** -0.5
        w[name] = z
    most = max([x["mlp"]["router"]["experts"] for x in cfg["layers"] if x["mlp"]["kind"] == "moe"], default=0)
    if most:
        order = torch.rand((cfg["vocab"], most), generator=g, device="cuda").argsort(1)
        w["embed"][:, :most] = torch.linspace(-2.0, 2.0, most, device="cuda")[order]
        for name, x in w.items():
            leaf = name.split(".", 1)[-1]
            if leaf in ("mix.o", "norm1") or leaf.endswith("down"):
                x[:most] = 0.0
            elif leaf == "mlp.router":
                x.zero_()
                x[torch.arange(len(x), device="cuda"), torch.randperm(most, generator=g, device="cuda")[:len(x)]] = 3.0
    return {name: x.to(torch.bfloat16) for name, x in w.items()}


def _write_model(path, cfg, w):
    with open(os.path.join(path, "config.json"), "w") as f:
        json.dump(cfg, f)
    head, at = {}, 0
    for name, x in w.items():
        n = x.numel() * 2
        head[name] = {"dtype": "BF16", "shape": list(x.shape), "data_offsets": [at, at + n]}
        at += n
    text = json.dumps(head).encode()
    data = torch.cat([x.reshape(-1) for x in w.values()]).view(torch.int16).cpu().numpy()
    with open(os.path.join(path, "model.safetensors"), "wb") as f:
        f.write(struct.pack("<Q", len(text)) + text)
        data.tofile(f)


def _prepare_model(case, seed):
    lib, model = kx(), C.c_void_p()
    context = case["prompt"] + case["steps"]
    if case["design"] == "kimi":
        cfg = _kimi_config(case, seed)
        check(lib.kx_model_create(C.byref(cfg), C.byref(model)))
    else:
        o, cfg = KxOpenOptions(), _hybrid_config(case)
        check(lib.kx_open_options_default(C.byref(o)))
        o.dtype, o.max_batch, o.max_context = DTYPES[case["dtype"]], case["batch"], context
        path = tempfile.mkdtemp(prefix="model_", dir="/dev/shm" if os.path.isdir("/dev/shm") else None)
        try:
            _write_model(path, cfg, _hybrid_weights(cfg, seed))
            check(lib.kx_model_open(path.encode(), C.byref(o), C.byref(model)))
        finally:
            shutil.rmtree(path, ignore_errors=True)
    held = _Held(model, lib.kx_model_destroy)
    ids = _ids(case, seed)
    s = {"case": case, "model": held, "prompt": np.ascontiguousarray(ids[:, :case["prompt"]]),
         "next": np.ascontiguousarray(ids[:, case["prompt"]:].T), "at": 0}
    if case["design"] == "kimi":
        # prompts in long steps; of a model with MoE layers token by token, the path whose tokens do not depend on how it is run
        check(lib.kx_model_set_prefill_chunk(model, 1 if case["moe_layers"] else 2048))
        if case["steps"]:          # the conversation so far
            check(lib.kx_prefill(model, s["prompt"].ctypes.data, case["batch"], case["prompt"]))
    return s


def _places(case):
    """Where a prompt's logits are asked for: of a scored prompt (kagalorn, rapitar) also in the middle."""
    return [case["prompt"] - 1] if case["design"] == "kimi" else [case["prompt"] // 2, case["prompt"] - 1]


def _run_model(s):
    case, lib, m, batch = s["case"], kx(), s["model"].h, s["case"]["batch"]
    if not case["steps"] and case["design"] != "kimi":
        places = np.array(_places(case), np.int32)
        out = np.empty((len(places), batch, case["vocab"]), np.float32)
        check(lib.kx_restart(m, batch))
        check(lib.kx_extend(m, s["prompt"].ctypes.data, case["prompt"], places.ctypes.data, len(places), out.ctypes.data))
        return out
    if case["steps"] and case["design"] == "kimi":
        check(lib.kx_model_rewind(m, s["at"]))     # the steps of the pass before are taken back
    else:
        check(lib.kx_prefill(m, s["prompt"].ctypes.data, batch, case["prompt"]))
    for row in s["next"]:
        check(lib.kx_decode_step(m, row.ctypes.data))
    s["at"] = case["steps"]
    out = np.empty((1, batch, case["vocab"]), np.float32)
    check(lib.kx_model_logits(m, out.ctypes.data))
    return out


def prepare(case, seed):
    return {"moe": _prepare_moe, "mla": _prepare_mla, "model": _prepare_model}[case["kind"]](case, seed)


def run(state):
    return {"moe": _run_moe, "mla": _run_mla, "model": _run_model}[state["case"]["kind"]](state)


# ---- what a pass cannot do without -----------------------------------------------------------------------------------
def _used(tokens, skewed):
    """Experts that `tokens` tokens meet, by the layer's distribution of logits and bias."""
    r = np.random.default_rng(7)
    score = 1 / (1 + np.exp(-r.standard_normal((tokens, E)))) + (-0.1 * np.log(np.arange(E) + 1.0) if skewed else 0.0)
    return len(np.unique(np.argpartition(-score, TOP, axis=1)[:, :TOP]))


_EXPERT = 3 * INTER * HIDDEN           # weights; packed and with their scales 4.5 bits each


def _kimi_layer(case):
    """(weights of a layer's attention, of its dense feed-forward)"""
    w, h = case["width"], case["heads"]
    return w * (Q_RANK + KV_RANK + ROPE) + h * (NOPE + ROPE) * Q_RANK + h * (NOPE + VHEAD) * KV_RANK + w * h * VHEAD, 3 * case["ff"] * w


def work(case):
    if case["kind"] == "moe":
        t = case["tokens"]
        moved = _used(t, case["path"] == "prompt") * _EXPERT * 4.5 / 8 + 2 * (_EXPERT + E * HIDDEN) + 3 * t * HIDDEN * 2
        return {"bytes": moved, "flops": 2.0 * t * ((TOP + 1) * _EXPERT + E * HIDDEN)}
    if case["kind"] == "mla":
        b, n = case["batch"], case["context"]
        return {"bytes": b * n * (KV_RANK + ROPE) * 2 + b * 64 * ((KV_RANK + ROPE) * 4 + KV_RANK * 2), "flops": 2.0 * b * n * 64 * (2 * KV_RANK + ROPE)}
    b, p, n, w = case["batch"], case["prompt"], case["steps"], case["width"]
    size = 4 if case["dtype"] == "float32" else 2
    logits = (2 if not n and case["design"] != "kimi" else 1) * b * case["vocab"]
    if case["design"] == "kimi":
        attn, dense = _kimi_layer(case)
        layers, moe = case["layers"], case["moe_layers"]
        met = layers * attn + (layers - moe) * dense + moe * ((TOP + 1) * _EXPERT + E * w)       # weights a token meets
        read = 2 * (layers * attn + (layers - moe) * dense) + moe * (_used(b, False) * _EXPERT * 4.5 / 8 + 2 * (_EXPERT + E * w))
        head, row = case["vocab"] * w, (KV_RANK + ROPE) * 2 * layers
        pair = 2.0 * case["heads"] * (NOPE + ROPE + VHEAD) * layers                               # a query and a key, expanded
        step = 2.0 * case["heads"] * (2 * KV_RANK + ROPE) * layers
        if not n:
            return {"bytes": read + 2 * head + b * p * (row + 2 * w) + 4 * logits, "flops": b * (2.0 * p * met + pair * p * (p + 1) / 2) + 2.0 * b * head}
        return {"bytes": n * (read + 2 * head + b * (p + n / 2) * row) + 4 * logits, "flops": n * b * (2.0 * (met + head) + step * (p + n / 2))}
    met = held = state = pairs = 0     # weights a token meets and that are read for many; state of a sequence; products of a sequence's attention
    total = p + n
    cfg = _hybrid_config(case)
    for layer in cfg["layers"]:
        m, f = layer["mixer"], layer["mlp"]
        h = m["heads"]
        if layer["type"] == "attention":
            mix = w * 128 * (3 * h + 2 * m["kv_heads"])
            keys = min(total, 1024) + max(0, total - 1024) / 16
            state += 2 * m["kv_heads"] * 128 * size * keys
            pairs += 4.0 * h * 128 * keys * total * 0.75
        elif layer["type"] == "delta":
            mix = w * (128 * (2 * m["kv_heads"] + 3 * h) + 2 * h)
            state += 2 * h * 128 * 128 * 4
            pairs += 6.0 * h * 128 * 128 * total
        elif layer["type"] == "mamba2":
            inner = h * m["vdim"]
            mix = w * (3 * inner + 2 * m["groups"] * m["state"] + h)
            state += 2 * inner * m["state"] * 4
            pairs += 4.0 * inner * m["state"] * total
        elif layer["type"] == "wkv":
            hd = h * m["dim"]
            mix = 5 * w * hd + 64 * (w + hd)
            state += 2 * hd * m["dim"] * 4
            pairs += 4.0 * hd * m["dim"] * total
        else:
            mix = w * (m["q_rank"] + 512 + 64 + 2 * h * 128) + m["q_rank"] * h * 192 + 512 * h * 256
            state += total * (512 + 64) * size
            pairs += h * (192 + 128) * total * (total + 1.0)
        gated = f["kind"] == "moe" or cfg["architecture"] == "Kagalorn"
        ff = 8 * f["expert"]["ff"] if f["kind"] == "moe" else f["ff"]
        met += mix + (3 if gated else 2) * w * ff
        more = min(64, 8 * b) / 8 if f["kind"] == "moe" else 1
        held += mix + (3 if gated else 2) * w * ff * more
        if f["kind"] == "moe":
            met += 64 * w
            held += 64 * w
    head = case["vocab"] * w
    prompt = {"bytes": size * (held + head) + b * (state + 4 * w * p) + 4 * logits, "flops": b * (2.0 * p * met + pairs) + 2.0 * head * b}
    if not n:
        return prompt
    return {"bytes": prompt["bytes"] + n * (size * (held + head) + b * state), "flops": prompt["flops"] + n * 2.0 * b * (met + head)}


def tolerance(case):
    """About four times the distance from exact() that was measured: 0.0047 (moe), 0.006 (mla), 0.009 (kimi), 0.004 (kagalorn,
    rapitar), 2e-6 in 32 bits; a choice of expert that rounding decides moves a kimi model with MoE layers further."""
    if case["kind"] == "moe":
        return {"rel": 1.6e-2, "max": 1.6e-1}
    if case["kind"] == "mla":
        return {"rel": 2e-2, "max": 2e-1}
    if case["dtype"] == "float32":
        return {"rel": 1e-5, "max": 1e-4}
    rel = 2.8e-2 if case["design"] == "kimi" else 1.6e-2
    return {"rel": rel, "max": 10 * rel}


# ---- the same in 64 bits -----------------------------------------------------------------------------------------------
def _rms(x, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps)


def _silu(x):
    return x * torch.sigmoid(x)


def _unpack(packed, scale):
    """INT4, eight to a word, lowest nibble first, q + 8; groups of 32 columns."""
    shift = torch.arange(0, 32, 4, device=packed.device, dtype=torch.int32)
    q = ((packed.unsqueeze(-1) >> shift) & 15).double().sub_(8.0).flatten(1)
    return q * scale.double().repeat_interleave(32, 1)


def _exact_routed(n, w, bias, experts, shared):
    """The routed layer's sum for rows n; experts(e) and shared give (gate, up, down)."""
    score = torch.sigmoid(n @ w.double().T)
    ids = (score + bias.double()).topk(TOP, 1).indices
    weight = score.gather(1, ids)
    weight = weight / weight.sum(1, keepdim=True) * SCALE
    ffn = lambda x, m: (_silu(x @ m[0].T) * (x @ m[1].T)) @ m[2].T
    out = ffn(n, shared)
    for e in ids.unique().tolist():
        tok, slot = (ids == e).nonzero(as_tuple=True)
        out.index_add_(0, tok, ffn(n[tok], experts(e)) * weight[tok, slot].unsqueeze(1))
    return out


def _exact_moe(case, seed):
    w, n, x = _moe_inputs(case, seed)
    expert = lambda e: [_unpack(w[k + "_packed"][e], w[k + "_scale"][e]) for k in ("gate", "up", "down")]
    shared = [w["shared_" + k].double() for k in ("gate", "up", "down")]
    return x.double() + _exact_routed(n.double(), w["router_gate"], w["router_bias"], expert, shared)


def _mla_scale():
    m = 0.1 * math.log(32.0) + 1.0                     # YaRN, factor 32
    return (NOPE + ROPE) ** -0.5 * m * m


def _exact_mla(case, seed):
    cache, q = _mla_inputs(case, seed)
    out = []
    for b in range(case["batch"]):
        top = torch.full((64, 1), -math.inf, device="cuda", dtype=torch.float64)
        z, o = torch.zeros_like(top), torch.zeros((64, KV_RANK), device="cuda", dtype=torch.float64)
        for rows in cache[b].split(16384):
            k = rows.double()
            s = q[b].double() @ k.T * _mla_scale()
            new = torch.maximum(top, s.max(1, keepdim=True).values)
            e, old = torch.exp(s - new), torch.exp(top - new)
            top, z, o = new, z * old + e.sum(1, keepdim=True), o * old + e @ k[:, :KV_RANK]
        out.append(o / z)
    return torch.stack(out)


# the values of random-init tensors: f(seed, tensor id, index), documented in kx.h as reproducible from these three
_GOLD, _M1, _M2, _U64 = 0x9E3779B97F4A7C15, 0xBF58476D1CE4E5B9, 0x94D049BB133111EB, (1 << 64) - 1


def _signed(v):
    v &= _U64
    return v - (1 << 64) if v >> 63 else v


def _mix(z):
    shr = lambda v, k: (v >> k) & ((1 << (64 - k)) - 1)
    z = (z ^ shr(z, 30)) * _signed(_M1)
    z = (z ^ shr(z, 27)) * _signed(_M2)
    return z ^ shr(z, 31)


def _key(seed, tid):
    z = (seed * _GOLD + tid + 1) & _U64
    z = ((z ^ (z >> 30)) * _M1) & _U64
    z = ((z ^ (z >> 27)) * _M2) & _U64
    return z ^ (z >> 31)


def _draws(key, at):
    return _mix((at + 1) * _signed(_GOLD) + _signed(key))


def _fill(seed, tid, shape, sigma, mean=0.0, first=0, magnitude=False, dtype=torch.bfloat16, device="cuda"):
    """Sum of twelve 16-bit uniforms, centred; `first`: index of the first element."""
    n, key = int(np.prod(shape)), _key(seed, tid)
    out = torch.empty(n, dtype=dtype, device=device)
    step = torch.tensor(sigma, dtype=torch.float32) * 2.0 ** -16
    for at in range(0, n, 1 << 24):
        i = torch.arange(first + at, first + min(n, at + (1 << 24)), device=device, dtype=torch.int64) * 3
        s = torch.zeros_like(i)
        for j in range(3):
            h = _draws(key, i + j)
            s += (h & 0xffff) + ((h >> 16) & 0xffff) + ((h >> 32) & 0xffff) + ((h >> 48) & 0xffff)
        z = mean + (s - 393210).float() * step.item()
        out[at:at + len(i)] = z.abs() if magnitude else z
    return out.view(shape)


def _words(seed, tid, shape, first, device="cuda"):
    n = int(np.prod(shape))
    i = torch.arange(first, first + n, device=device, dtype=torch.int64)
    return ((_draws(_key(seed, tid), i >> 1) >> ((i & 1) * 32)) & 0xffffffff).to(torch.int32).view(shape)


def _yarn():
    """Rotation frequencies of ROPE / 2 pairs: theta 50000, factor 32, original context 4096, ramp between 32 and 1 turns."""
    f = 50000.0 ** (-torch.arange(0, ROPE, 2, device="cuda", dtype=torch.float64) / ROPE)
    edge = lambda turns: ROPE * math.log(4096 / (turns * 2 * math.pi)) / (2 * math.log(50000.0))
    low, high = max(math.floor(edge(32)), 0), min(math.ceil(edge(1)), ROPE - 1)
    ramp = ((torch.arange(ROPE // 2, device="cuda", dtype=torch.float64) - low) / (high - low)).clamp(0, 1)
    return f / 32.0 * ramp + f * (1 - ramp)


def _softmax_rows(q, k, v, seen, more=None):
    """softmax(q k^T) v for rows of queries; `seen`: bool [queries][keys]; `more`: a score that only the denominator has."""
    s = (q @ k.T).masked_fill_(~seen, -math.inf)
    top = s.max(1, keepdim=True).values
    if more is not None:
        top = top.clamp(min=more)
    e = torch.exp(s - top)
    z = e.sum(1, keepdim=True) + (0.0 if more is None else torch.exp(more - top))
    return e @ v / z


def _exact_kimi(case, seed):
    c, ids = _kimi_config(case, seed), torch.from_numpy(_ids(case, seed).astype(np.int64)).cuda()
    w, heads, (batch, total) = case["width"], case["heads"], ids.shape
    norm = lambda tid, n: _fill(seed, tid, (n,), 0.02, 1.0).double()
    mat = lambda tid, r, k: _fill(seed, tid, (r, k), 0.02).double()
    x = torch.stack([_fill(seed, 1, (w,), 1.0, first=t * w) for t in ids.unique().tolist()])
    x = x[torch.searchsorted(ids.unique(), ids.reshape(-1))].double()          # [batch * total][w]
    angle = torch.arange(total, device="cuda", dtype=torch.float64).unsqueeze(1) * _yarn()
    cos, sin = angle.cos(), angle.sin()

    def turn(v):                   # [total][...][ROPE], pairs of neighbours
        a, b, cs, sn = v[..., 0::2], v[..., 1::2], cos, sin
        if v.dim() == 3:
            cs, sn = cos.unsqueeze(1), sin.unsqueeze(1)
        return torch.cat([a * cs - b * sn, b * cs + a * sn], -1)

    seen = torch.ones((total, total), dtype=torch.bool, device="cuda").tril_()
    for l in range(case["layers"]):
        b = (l + 1) * 64
        n = _rms(x, c.rms_eps) * norm(b, w)
        qa = _rms(n @ mat(b + 1, Q_RANK, w).T, c.rms_eps) * norm(b + 2, Q_RANK)
        q = (qa @ mat(b + 3, heads * (NOPE + ROPE), Q_RANK).T).view(batch, total, heads, NOPE + ROPE)
        kva = n @ mat(b + 4, KV_RANK + ROPE, w).T
        lat = _rms(kva[:, :KV_RANK], c.rms_eps) * norm(b + 5, KV_RANK)
        kv = (lat @ mat(b + 6, heads * (NOPE + VHEAD), KV_RANK).T).view(batch, total, heads, NOPE + VHEAD)
        att = torch.empty((batch, total, heads, VHEAD), dtype=torch.float64, device="cuda")
        for s in range(batch):
            kr, qr = turn(kva.view(batch, total, -1)[s, :, KV_RANK:]), turn(q[s, :, :, NOPE:])
            for h in range(heads):
                qh = torch.cat([q[s, :, h, :NOPE], qr[:, h]], 1) * _mla_scale()
                att[s, :, h] = _softmax_rows(qh, torch.cat([kv[s, :, h, :NOPE], kr], 1), kv[s, :, h, NOPE:], seen)
        x = x + att.view(batch * total, -1) @ mat(b + 7, w, heads * VHEAD).T
        n = _rms(x, c.rms_eps) * norm(b + 8, w)
        if l < c.first_dense:
            ff = case["ff"]
            x = x + (_silu(n @ mat(b + 9, ff, w).T) * (n @ mat(b + 10, ff, w).T)) @ mat(b + 11, w, ff).T
            continue
        tensors = ((14, INTER, w), (16, INTER, w), (18, w, INTER))

        def expert(e):
            return [_unpack(_words(seed, b + t, (r, k // 8), e * r * k // 8), _fill(seed, b + t + 1, (r, k // 32), 0.02, first=e * r * k // 32, magnitude=True))
                    for t, r, k in tensors]

        x = x + _exact_routed(n, _fill(seed, b + 12, (E, w), w ** -0.5), _fill(seed, b + 13, (E,), 0.01, dtype=torch.float32), expert,
                              [mat(b + 20, INTER, w), mat(b + 21, INTER, w), mat(b + 22, w, INTER)])
    x = x.view(batch, total, w)[:, -1]
    return ((_rms(x, c.rms_eps) * norm(2, w)) @ mat(3, case["vocab"], w).T).unsqueeze(0)


def _conv(x, kernel, bias=None):
    """Causal convolution along the positions, x [batch][n][channels], kernel [channels][taps]; the last tap meets the present."""
    taps, n = kernel.shape[1], x.shape[1]
    x = torch.cat([x.new_zeros((x.shape[0], taps - 1, x.shape[2])), x], 1)
    y = sum(x[:, j:j + n] * kernel[:, j] for j in range(taps))
    return _silu(y if bias is None else y + bias)


def _attention(h, w, m):
    (b, n, _), heads, kv = h.shape, m["heads"], m["kv_heads"]
    q = (_rms(h @ w("q").T, 1e-5) * w("q.norm")).view(b, n, heads, -1) * m["scale"]
    k = (_rms(h @ w("k").T, 1e-5) * w("k.norm")).view(b, n, kv, -1)
    v = (h @ w("v").T).view(b, n, kv, -1)
    size, pool = m["mask"]["size"], m["mask"]["pool"]
    i, nb = torch.arange(n, device="cuda").unsqueeze(1), n // pool
    j, e = torch.arange(n, device="cuda").unsqueeze(0), torch.arange(nb, device="cuda").unsqueeze(0) * pool + pool - 1
    seen = torch.cat([(j <= i) & (j > i - size), e <= i - size], 1)
    means = lambda t: torch.cat([t, t[:, :nb * pool].view(b, nb, pool, kv, -1).mean(2)], 1)
    k, v, o = means(k), means(v), torch.empty((b, n, heads, m["vdim"]), dtype=torch.float64, device="cuda")
    for s in range(b):
        for a in range(heads):
            o[s, :, a] = _softmax_rows(q[s, :, a], k[s, :, a * kv // heads], v[s, :, a * kv // heads], seen, torch.zeros((), dtype=torch.float64, device="cuda"))
    return (o.view(b, n, -1) * torch.sigmoid(h @ w("g").T)) @ w("o").T


def _delta(h, w, m):
    (b, n, _), heads, kv, dim = h.shape, m["heads"], m["kv_heads"], m["dim"]
    q, k, v = (_conv(h @ w(c).T, w(c + ".conv")) for c in "qkv")
    unit = lambda t: t * torch.rsqrt(t.square().sum(-1, keepdim=True) + 1e-6)
    q = unit(q.view(b, n, kv, dim)).repeat_interleave(heads // kv, 2) * dim ** -0.5
    k = unit(k.view(b, n, kv, dim)).repeat_interleave(heads // kv, 2)
    v, beta = v.view(b, n, heads, -1), torch.sigmoid(h @ w("b").T)
    decay = torch.exp(-torch.exp(w("A_log")) * torch.nn.functional.softplus(h @ w("a").T + w("dt_bias"), threshold=700))
    s, o = v.new_zeros((b, heads, dim, v.shape[-1])), torch.empty_like(v)
    for t in range(n):
        s = s * decay[:, t, :, None, None]
        u = beta[:, t, :, None] * (v[:, t] - (s * k[:, t].unsqueeze(-1)).sum(2))
        s = s + k[:, t].unsqueeze(-1) * u.unsqueeze(2)
        o[:, t] = (s * q[:, t].unsqueeze(-1)).sum(2)
    return ((_rms(o, 1e-5) * w("norm")).view(b, n, -1) * _silu(h @ w("g").T)) @ w("o").T


def _mamba2(h, w, m):
    (b, n, _), heads, state, groups = h.shape, m["heads"], m["state"], m["groups"]
    inner = heads * m["vdim"]
    z, x, dt = (h @ w("in").T).split([inner, inner + 2 * groups * state, heads], 2)
    x, bs, cs = _conv(x, w("conv"), w("conv.b")).split([inner, groups * state, groups * state], 2)
    x = x.view(b, n, heads, -1)
    bs, cs = (t.view(b, n, groups, state).repeat_interleave(heads // groups, 2) for t in (bs, cs))
    dt = torch.nn.functional.softplus(dt + w("dt_bias"), threshold=700)
    decay = torch.exp(-torch.exp(w("A_log")) * dt)
    s, y = x.new_zeros((b, heads, state, m["vdim"])), torch.empty_like(x)
    for t in range(n):
        s = s * decay[:, t, :, None, None] + (bs[:, t] * dt[:, t, :, None]).unsqueeze(-1) * x[:, t].unsqueeze(2)
        y[:, t] = (s * cs[:, t].unsqueeze(-1)).sum(2)
    y = (y + w("D")[:, None] * x).view(b, n, inner) * _silu(z)
    return (_rms(y.view(b, n, m["norm_groups"], -1), 1e-5).view(b, n, inner) * w("norm")) @ w("o").T


def _wkv(h, w, m):
    (b, n, _), heads = h.shape, m["heads"]
    before = torch.cat([torch.zeros_like(h[:, :1]), h[:, :-1]], 1)
    mix = {c: h + (before - h) * w("mu." + c) for c in "rkvgw"}
    r, k, v = ((mix[c] @ w(c).T).view(b, n, heads, -1) for c in "rkv")
    decay = torch.exp(-torch.exp(torch.tanh(mix["w"] @ w("w1").T) @ w("w2").T + w("w0"))).view(b, n, heads, -1)
    s, o, u = v.new_zeros((b, heads, m["dim"], m["dim"])), torch.empty_like(v), w("u").unsqueeze(-1)
    for t in range(n):
        kv = k[:, t].unsqueeze(-1) * v[:, t].unsqueeze(2)
        o[:, t] = ((s + u * kv) * r[:, t].unsqueeze(-1)).sum(2)
        s = s * decay[:, t].unsqueeze(-1) + kv
    return ((_rms(o, 1e-5).view(b, n, -1) * w("norm")) * _silu(mix["g"] @ w("g").T)) @ w("o").T


def _latent(h, w, m):
    (b, n, _), heads, dim, dims = h.shape, m["heads"], m["dim"], m["rot"]["dims"]
    a = torch.arange(n, device="cuda", dtype=torch.float64).unsqueeze(1) * m["rot"]["base"] ** (-2.0 * torch.arange(dims // 2, device="cuda", dtype=torch.float64) / dims)
    cos, sin = a.cos(), a.sin()

    def turn(t, cs, sn):           # dimension i and i + dims / 2
        u, v = t[..., :dims // 2], t[..., dims // 2:dims]
        return torch.cat([u * cs - v * sn, v * cs + u * sn, t[..., dims:]], -1)

    q = ((_rms(h @ w("dq").T, 1e-5) * w("dq.norm")) @ w("uq").T).view(b, n, heads, -1)
    q = torch.cat([q[..., :dim], turn(q[..., dim:], cos.unsqueeze(1), sin.unsqueeze(1))], -1) * m["scale"]
    c, shared = (h @ w("dkv").T).split([m["kv_rank"], m["rot_dim"]], 2)
    c, shared = _rms(c, 1e-5) * w("dkv.norm"), turn(shared, cos, sin)
    k, v = (c @ w("uk").T).view(b, n, heads, -1), (c @ w("uv").T).view(b, n, heads, -1)
    seen, o = torch.ones((n, n), dtype=torch.bool, device="cuda").tril_(), torch.empty_like(v)
    for s in range(b):
        for x in range(heads):
            o[s, :, x] = _softmax_rows(q[s, :, x], torch.cat([k[s, :, x], shared[s]], 1), v[s, :, x], seen, w("sink")[x])
    return (o.view(b, n, -1) * torch.sigmoid(h @ w("g").T)) @ w("o").T


def _experts(h, w, f):
    flat = h.reshape(-1, h.shape[-1])
    top, ids = (flat @ w("router").T + w("router.b")).topk(f["router"]["top"], 1)
    weight, out = torch.softmax(top, 1), torch.zeros_like(flat)
    for e in ids.unique().tolist():
        tok, slot = (ids == e).nonzero(as_tuple=True)
        y = (_silu(flat[tok] @ w(f"e{e}.gate").T) * (flat[tok] @ w(f"e{e}.up").T)) @ w(f"e{e}.down").T
        out.index_add_(0, tok, y * weight[tok, slot].unsqueeze(1))
    return out.view(h.shape)


def _exact_hybrid(case, seed):
    cfg = _hybrid_config(case)
    weights, ids = _hybrid_weights(cfg, seed), torch.from_numpy(_ids(case, seed).astype(np.int64)).cuda()
    under = lambda p: lambda name: weights[p + name].double()
    g, x = under(""), weights["embed"][ids].double()
    kinds = {"attention": _attention, "delta": _delta, "mamba2": _mamba2, "wkv": _wkv, "latent_attention": _latent}
    if case["design"] == "rapitar":
        for i, layer in enumerate(cfg["layers"]):
            h, mlp, f = _rms(x, 1e-5) * (1 + g(f"l{i}.norm1")), under(f"l{i}.mlp."), layer["mlp"]
            y = kinds[layer["type"]](h, under(f"l{i}.mix."), layer["mixer"])
            x = x + y + (_experts(h, mlp, f) if f["kind"] == "moe" else torch.nn.functional.gelu(h @ mlp("up").T, approximate="tanh") @ mlp("down").T)
        scale = 1 + g("final.norm")
        x = _rms(x, 1e-5)
    else:
        grouped = lambda t: _rms(t.view(*t.shape[:-1], 2, -1), 1e-5).view(t.shape)
        s = x.unsqueeze(0).repeat(cfg["streams"], 1, 1, 1)
        for i, layer in enumerate(cfg["layers"]):
            mlp = under(f"l{i}.mlp.")

            def glu(h):
                a, u = (h @ mlp("gate").T).clamp(max=7.0), (h @ mlp("up").T).clamp(-7.0, 7.0)
                return (a * torch.sigmoid(1.702 * a) * (u + 1)) @ mlp("down").T

            for q, f in ((1, lambda h: kinds[layer["type"]](h, under(f"l{i}.mix."), layer["mixer"])), (2, glu)):
                hc = under(f"l{i}.hc{q}.")
                y = f(grouped(torch.tensordot(hc("in"), s, 1)) * g(f"l{i}.norm{q}"))
                s = torch.tensordot(hc("mix").T, s, 1) + hc("out").view(-1, 1, 1, 1) * y
        x, scale = grouped(s.sum(0)), g("final.norm")
    places = [case["prompt"] + case["steps"] - 1] if case["steps"] else _places(case)
    return torch.stack([(x[:, p] * scale) @ g("head").T for p in places])


def exact(case, seed):
    if case["kind"] == "model":
        return (_exact_kimi if case["design"] == "kimi" else _exact_hybrid)(case, seed)
    return (_exact_moe if case["kind"] == "moe" else _exact_mla)(case, seed)
