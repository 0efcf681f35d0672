"""The work that a user of this library has it do, as measurable cases.

Four kinds of call, each through the Python entry points over device tensors:

* ``prefill`` -- attention of a prompt, an encoder's frames, or a chunk of a
  prompt over a KV cache (``flash_attention_forward`` where query and KV heads
  are as many and nothing is cached, ``attention_forward`` otherwise);
* ``decode``  -- one append-and-attend step of a batch of sequences over its
  KV cache (``KVCache.decode_step``);
* ``cross``   -- a few decoder queries over a long encoder memory
  (``attention_forward`` without a mask);
* ``qkv``     -- the q/k/v projections and rotary embedding of a decode step,
  for the layers of a model one after the other (``qkv_rope``).

Everything is float32, the library's only data type.
"""
import importlib.util
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "neural-network-engine_amd")
_DEV = "cuda:0"
_STEPS = 64            # decode steps between two resets of the cache lengths


def _package():
    if "nne_amd" not in sys.modules:
        spec = importlib.util.spec_from_file_location(
            "nne_amd", os.path.join(_PKG, "__init__.py"), submodule_search_locations=[_PKG])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["nne_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["nne_amd"]


def _prefill(b, hq, hkv, tq, tk, d, causal, std=1.0):
    return {"kind": "prefill", "b": b, "hq": hq, "hkv": hkv, "tq": tq, "tk": tk, "d": d,
            "causal": causal, "std": std}


def listed():
    return [
        # A short prompt on a small model: the call's latency is what counts.
        dict(_prefill(1, 4, 4, 256, 256, 64, True), name="prompt_small"),
        # One user's prompt (odd length) on a LLaMA-shaped layer: too little work to
        # fill the chip.
        dict(_prefill(1, 32, 8, 509, 509, 128, True), name="prompt_gqa"),
        # A batch of long prompts on a LLaMA-shaped layer, the ordinary prefill.
        dict(_prefill(4, 32, 8, 2048, 2048, 128, True), name="prefill_gqa"),
        # One very long prompt at head dim 64.
        dict(_prefill(1, 16, 16, 16384, 16384, 64, True, 0.5), name="prefill_long"),
        # The encoder layers of a Whisper batch: no mask, 1500 frames (not a multiple
        # of any tile).
        dict(_prefill(8, 20, 20, 1500, 1500, 64, False), name="encoder"),
        # The next chunk of a prompt over the rows a KV cache already holds, everything
        # ragged: 333 new rows over 3001, K/V read in place from the cache.
        dict(_prefill(2, 16, 4, 333, 3001, 128, True), name="prefill_chunk"),
        # Prefill at the wide head dims that some models use.
        dict(_prefill(1, 16, 16, 4096, 4096, 256, True), name="prefill_d256"),
        dict(_prefill(1, 16, 16, 4096, 4096, 512, True), name="prefill_d512"),
        # A decode step of a serving batch: 32 sequences of 512-4096 cached rows.
        {"kind": "decode", "name": "decode_batch", "b": 32, "hq": 32, "hkv": 8, "d": 128,
         "lo": 512, "hi": 4096},
        # A decode step of one user's sequence: the latency of a token.
        {"kind": "decode", "name": "decode_single", "b": 1, "hq": 32, "hkv": 8, "d": 128,
         "lo": 1733, "hi": 1733},
        # Eight decoder queries over 1500 encoder frames.
        {"kind": "cross", "name": "cross", "b": 8, "h": 20, "tq": 8, "tk": 1500, "d": 64},
        # The projections of a serving batch's decode step, three LLaMA-shaped layers
        # (302 MB of weights: more than any cache holds, as in a whole model).
        {"kind": "qkv", "name": "qkv", "b": 32, "c": 4096, "hq": 32, "hkv": 8, "d": 128,
         "layers": 3, "bias": False, "rope": True},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["prefill"] * 5 + ["decode"] * 3 + ["cross"] + ["qkv"])
    if kind == "prefill":
        d = rng.choice([64, 64, 64, 128, 128, 128, 80, 96, 192, 256, 512])
        hkv = rng.choice([1, 2, 4, 8, 12, 16, 20])
        g = rng.choice([1, 1, 1, 2, 4, 8])
        tq = _log_int(rng, 48, 8192)
        causal = rng.random() < 0.7
        # A quarter of the causal ones continue a cached prompt.
        tk = tq + (_log_int(rng, 16, 4096) if causal and rng.random() < 0.25 else 0)
        case = _prefill(1, hkv * g, hkv, tq, tk, d, causal, rng.choice([0.5, 1.0]))
        per = work(case)["flops"]
        while per > 4e11 and case["tq"] > 1024:
            case["tq"] //= 2
            case["tk"] //= 2
            per = work(case)["flops"]
        case["b"] = max(1, min(rng.choice([1, 1, 2, 3, 4, 8]), int(4e11 / per)))
        return case
    if kind == "decode":
        hkv = rng.choice([2, 4, 8, 12])
        g = rng.choice([1, 1, 4, 4, 8])
        hi = _log_int(rng, 64, 8192)
        b = min(_log_int(rng, 1, 64), max(1, 131072 // hi))
        return {"kind": "decode", "b": b, "hq": hkv * g, "hkv": hkv,
                "d": rng.choice([64, 128, 128]), "lo": max(1, hi // rng.choice([1, 2, 8])),
                "hi": hi}
    if kind == "cross":
        return {"kind": "cross", "b": rng.randint(1, 16), "h": rng.choice([6, 8, 12, 16, 20]),
                "tq": rng.choice([1, 1, 2, 4, 5, 8, 13]), "tk": _log_int(rng, 200, 3000),
                "d": 64}
    hkv, d = rng.choice([(4, 64), (8, 128), (12, 64), (8, 64)])
    g = rng.choice([1, 4])
    return {"kind": "qkv", "b": _log_int(rng, 1, 64), "c": hkv * g * d, "hq": hkv * g, "hkv": hkv,
            "d": d, "layers": rng.randint(1, 3), "bias": rng.random() < 0.5,
            "rope": rng.random() < 0.6}


def _randn(gen, *shape, std=1.0):
    return torch.randn(shape, generator=gen, device=_DEV, dtype=torch.float32) * std


def _inputs(case, seed):
    """The call's input tensors, from the seed alone (the same for run and exact)."""
    gen = torch.Generator(device=_DEV).manual_seed(seed)
    kind = case["kind"]
    if kind in ("prefill", "cross"):
        hq, hkv = (case["hq"], case["hkv"]) if kind == "prefill" else (case["h"], case["h"])
        b, tq, tk, d = case["b"], case["tq"], case["tk"], case["d"]
        std = case.get("std", 1.0)
        q = _randn(gen, b, hq, tq, d, std=std)
        # A chunk over a cache reads K and V in place from buffers with room for more rows.
        cap = tk if tq == tk or kind == "cross" else tk + 99
        k = _randn(gen, b, hkv, cap, d, std=std)
        v = _randn(gen, b, hkv, cap, d, std=std)
        # Real queries and keys differ in size from position to position.
        q *= torch.rand(tq, 1, generator=gen, device=_DEV) + 0.5
        k *= torch.rand(cap, 1, generator=gen, device=_DEV) + 0.5
        return {"q": q, "k": k[:, :, :tk], "v": v[:, :, :tk]}
    if kind == "decode":
        b, hq, hkv, d = case["b"], case["hq"], case["hkv"], case["d"]
        lens = np.random.default_rng(seed).integers(case["lo"], case["hi"] + 1, b).astype(np.int32)
        cap = case["hi"] + _STEPS
        k, v = _randn(gen, b, hkv, cap, d), _randn(gen, b, hkv, cap, d)
        # Rows that no step has written yet are empty.
        unused = torch.arange(cap, device=_DEV) >= torch.from_numpy(lens).to(_DEV)[:, None]
        k.masked_fill_(unused[:, None, :, None], 0.0)
        v.masked_fill_(unused[:, None, :, None], 0.0)
        return {"k": k, "v": v, "lens": lens, "q": _randn(gen, b, hq, 1, d),
                "k_new": _randn(gen, b, hkv, 1, d), "v_new": _randn(gen, b, hkv, 1, d)}
    b, c, hq, hkv, d = case["b"], case["c"], case["hq"], case["hkv"], case["d"]
    layers = []
    for _ in range(case["layers"]):
        w = [_randn(gen, h * d, c, std=1.0 / math.sqrt(c)) for h in (hq, hkv, hkv)]
        bias = [_randn(gen, h * d, std=0.1) if case["bias"] else None for h in (hq, hkv, hkv)]
        layers.append((w, bias))
    pos = np.random.default_rng(seed).integers(0, 4096, b).astype(np.int32)
    return {"x": _randn(gen, b, c), "layers": layers, "pos": pos}


def prepare(case, seed):
    nne = _package()
    t = _inputs(case, seed)
    state = {"case": case}
    if case["kind"] == "decode":
        cache = nne.KVCache(1, case["b"], case["hkv"], t["k"].shape[2], case["d"], device=_DEV)
        cache.k[0], cache.v[0] = t["k"], t["v"]
        cache.set_lengths(0, t["lens"])
        state.update(cache=cache, lens=t["lens"], q=t["q"], k_new=t["k_new"], v_new=t["v_new"],
                     step=0)
    elif case["kind"] == "qkv":
        hq, hkv, d = case["hq"], case["hkv"], case["d"]
        state.update(x=t["x"], layers=[(nne.qkv_pack(*w, hq, hkv), bias) for w, bias in t["layers"]],
                     rope=nne.RotaryEmbedding(d, 4096, device=_DEV) if case["rope"] else None,
                     pos_host=t["pos"], pos_dev=torch.from_numpy(t["pos"]).to(_DEV))
    else:
        state.update(t)
    return state


def run(state):
    nne, case = _package(), state["case"]
    kind = case["kind"]
    if kind == "prefill":
        if case["hq"] == case["hkv"] and case["tq"] == case["tk"]:
            return nne.flash_attention_forward(state["q"], state["k"], state["v"], case["causal"])
        return nne.attention_forward(state["q"], state["k"], state["v"], case["causal"],
                                     q_offset=case["tk"] - case["tq"])
    if kind == "cross":
        return nne.attention_forward(state["q"], state["k"], state["v"], False)
    if kind == "decode":
        cache = state["cache"]
        if state["step"] == _STEPS:     # the sequences have ended: others of their lengths
            cache.set_lengths(0, state["lens"])
            state["step"] = 0
        out = cache.decode_step(0, state["q"], state["k_new"], state["v_new"])
        state["step"] += 1
        return {"out": out, "k": cache.k[0], "v": cache.v[0], "lens": cache.lens_dev[0]}
    return [nne.qkv_rope(state["x"], packed, *bias, state["rope"], state["pos_dev"],
                         state["pos_host"], case["hq"], case["hkv"], head_dim=case["d"])
            for packed, bias in state["layers"]]


def work(case):
    kind = case["kind"]
    if kind in ("prefill", "cross"):
        hq, hkv = (case["hq"], case["hkv"]) if kind == "prefill" else (case["h"], case["h"])
        b, tq, tk, d = case["b"], case["tq"], case["tk"], case["d"]
        pairs = tq * tk
        if case.get("causal"):      # row r sees the first r + 1 + tk - tq keys
            pairs = tq * (tk - tq) + tq * (tq + 1) // 2
        return {"bytes": 4 * d * b * (2 * hq * tq + 2 * hkv * tk), "flops": 4 * b * hq * pairs * d}
    if kind == "decode":
        b, hq, hkv, d = case["b"], case["hq"], case["hkv"], case["d"]
        rows = b * ((case["lo"] + case["hi"]) / 2 + 1)      # cached rows and the new one
        return {"bytes": 4 * d * (2 * hkv * rows + 2 * b * hq + 2 * b * hkv),
                "flops": 4 * hq * rows * d}
    n = (case["hq"] + 2 * case["hkv"]) * case["d"]
    b, c = case["b"], case["c"]
    return {"bytes": 4 * case["layers"] * (n * c + b * c + b * n),
            "flops": 2 * case["layers"] * b * c * n}


def tolerance(case):
    # Float32 throughout: a projection's sums of c products, attention's of d products
    # (whose rounding the exponential carries into the weights) and of up to 16384 weights.
    # About four times the errors measured against 64 bits (5.2e-7 and up to 1.1e-6).
    if case["kind"] == "qkv":
        return {"rel": 2e-6, "max": 2e-5}
    return {"rel": 5e-6, "max": 1e-4}


def _attend(q, k, v, causal, offset):
    """Plain softmax attention of one KV head in 64 bits: q [G, Tq, d], k and v [Tk, d]."""
    k, v = k.double(), v.double()
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    block = max(1, (1 << 27) // max(1, k.shape[0]))
    for g in range(q.shape[0]):
        for r in range(0, q.shape[1], block):
            s = q[g, r:r + block].double() @ k.T / math.sqrt(q.shape[2])
            if causal:
                rows = torch.arange(r, r + s.shape[0], device=q.device)[:, None]
                s.masked_fill_(torch.arange(s.shape[1], device=q.device) > rows + offset, -math.inf)
            out[g, r:r + block] = torch.softmax(s, -1) @ v
    return out


def _rotation(pos, d):
    """cos and sin [B, 1, 1, d] of the rotary embedding at positions pos.  The tables are
    data in 32 bits, so every step up to them is rounded there: theta^(2i/d), its
    reciprocal, the angle, and its cosine and sine."""
    f = np.float32
    power = np.power(1e4, (f(2) * np.arange(d // 2, dtype=f) / f(d)).astype(np.float64)).astype(f)
    angle = (pos.astype(f)[:, None] * (f(1) / power)).astype(np.float64)
    return (torch.from_numpy(np.tile(fn(angle).astype(f), 2)).double().to(_DEV)[:, None, None]
            for fn in (np.cos, np.sin))


def exact(case, seed):
    t = _inputs(case, seed)
    kind = case["kind"]
    if kind in ("prefill", "cross"):
        q, k, v = t["q"], t["k"], t["v"]
        g = q.shape[1] // k.shape[1]
        out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
        for b in range(q.shape[0]):
            for h in range(k.shape[1]):
                out[b, h * g:(h + 1) * g] = _attend(q[b, h * g:(h + 1) * g], k[b, h], v[b, h],
                                                    case.get("causal", False),
                                                    case["tk"] - case["tq"])
        return out
    if kind == "decode":
        lens = t["lens"]
        rows, at = torch.arange(case["b"], device=_DEV), torch.from_numpy(lens).long().to(_DEV)
        k, v = t["k"], t["v"]
        k[rows, :, at] = t["k_new"][:, :, 0]
        v[rows, :, at] = t["v_new"][:, :, 0]
        g = case["hq"] // case["hkv"]
        out = torch.empty(t["q"].shape, dtype=torch.float64, device=_DEV)
        for b in range(case["b"]):
            n = int(lens[b]) + 1
            for h in range(case["hkv"]):
                out[b, h * g:(h + 1) * g] = _attend(t["q"][b, h * g:(h + 1) * g], k[b, h, :n],
                                                    v[b, h, :n], False, 0)
        return {"out": out, "k": k.double(), "v": v.double(), "lens": at + 1}
    cos, sin = _rotation(t["pos"], case["d"])
    outs = []
    for w, bias in t["layers"]:
        layer = []
        for i, (wi, bi) in enumerate(zip(w, bias)):
            y = t["x"].double() @ wi.double().T
            if bi is not None:
                y = y + bi.double()
            y = y.view(case["b"], -1, 1, case["d"])
            if case["rope"] and i < 2:
                half = case["d"] // 2
                y = y * cos + torch.cat([-y[..., half:], y[..., :half]], -1) * sin
            layer.append(y)
        outs.append(tuple(layer))
    return outs
