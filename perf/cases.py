"""The work a user of this framework has it do, as timed cases.

Every case goes through the public classes (``TurboPolarKVCacheRuntime``,
``TurboPolarFastCache``, ``HipKernelBridge``, ``QJLResidualEncoder``), over the
range of shapes that the configurations, the tests and the benchmark of this
repository use: contexts from one page to 131,072 tokens, 1 to 32 kv heads,
query-head groups of 1 to 20, batches, every page layout, fp16 and fp32 inputs.

``op`` names what one pass does:

* ``attend``   one decode step's attention over a cache that holds ``tokens``
  tokens (whole pages plus the dense tail), as a serving loop calls it;
* ``prefill``  a prompt of ``tokens`` tokens appended to a new cache (encode);
* ``fetch``    a prompt fed to a new cache in chunks, each returning the whole
  history decompressed (the prefill path of the model hook);
* ``generate`` a short prompt and then ``steps`` single-token decode steps on a
  new cache (append, page flushes and attention);
* ``scores``   the fused dequantise-and-score call over every stored token;
* ``qjl``      residual sketches of every stored token, the query's sketch and
  the attention step that uses both.
"""

import math

import torch

from turbopolar_amd import HipKernelBridge, TurboPolarConfig, TurboPolarFastCache, TurboPolarKVCacheRuntime
from turbopolar_amd.qjl import QJLResidualEncoder, qjl_projection

PAGE, DIM, PAIRS = 64, 128, 64

# int8 log radii, level-1 bits, deep bits, split: the configuration's defaults,
# the layout of make_turbo_caches, and other widths that the configuration takes.
LAYOUTS = {
    "default": (False, 4, 4, 64),
    "fast": (True, 4, 8, 0),
    "deep2": (False, 4, 2, 64),
    "l1_8bit": (False, 8, 4, 32),
    "odd_split": (True, 4, 2, 46),
    "int8_angles4": (True, 4, 4, 64),
}


def listed():
    return [
        # A chat turn's early decode step: 1,000 tokens, where latency counts.
        {"name": "attend_1k", "op": "attend", "layout": "default", "batch": 1, "hq": 32, "hkv": 8, "tokens": 1000},
        # The benchmark's own shape, between two page flushes.
        {"name": "attend_32k", "op": "attend", "layout": "default", "batch": 1, "hq": 32, "hkv": 8, "tokens": 32805},
        # The largest context, 8 query heads a group, in the layout of make_turbo_caches.
        {"name": "attend_131k", "op": "attend", "layout": "fast", "batch": 1, "hq": 64, "hkv": 8, "tokens": 131072},
        # A serving batch of middling contexts.
        {"name": "attend_batch", "op": "attend", "layout": "default", "batch": 16, "hq": 32, "hkv": 8, "tokens": 4000},
        # No query grouping: one query head per kv head.
        {"name": "attend_mha", "op": "attend", "layout": "fast", "batch": 1, "hq": 32, "hkv": 32, "tokens": 9000},
        # 2-bit deep angles, the most compressed keys the configuration takes.
        {"name": "attend_deep2", "op": "attend", "layout": "deep2", "batch": 1, "hq": 32, "hkv": 8, "tokens": 16400},
        # Scores alone, over a whole 32k cache.
        {"name": "scores_32k", "op": "scores", "layout": "default", "batch": 1, "hq": 32, "hkv": 8, "tokens": 32768},
        # A long prompt compressed at once.
        {"name": "prefill_32k", "op": "prefill", "layout": "default", "batch": 1, "hkv": 8, "tokens": 32773,
         "dtype": "float16"},
        # A float32 model's prompt, in the layout of make_turbo_caches.
        {"name": "prefill_f32", "op": "prefill", "layout": "fast", "batch": 1, "hkv": 8, "tokens": 6100,
         "dtype": "float32"},
        # Chunked prefill through the model hook's cache.
        {"name": "fetch_8k", "op": "fetch", "layout": "fast", "batch": 1, "hkv": 8, "tokens": 8100, "chunk": 2048},
        # Token by token generation on one layer's cache.
        {"name": "generate", "op": "generate", "layout": "fast", "batch": 1, "hq": 32, "hkv": 8, "tokens": 300,
         "steps": 40},
        # The residual-sketch correction, sketches made and used.
        {"name": "qjl_8k", "op": "qjl", "layout": "default", "batch": 1, "hq": 32, "hkv": 8, "tokens": 8192},
    ]


# (query heads, kv heads) of the configurations, the tests and the benchmark.
HEADS = [(32, 8), (64, 8), (32, 32), (8, 8), (28, 4), (40, 8), (4, 1), (8, 1), (16, 4), (24, 2), (40, 2), (8, 2)]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["attend"] * 5 + ["prefill"] * 3 + ["scores", "fetch", "generate", "qjl"])
    layout = rng.choice(["default"] * 3 + ["fast"] * 3 + ["deep2", "l1_8bit", "odd_split", "int8_angles4"])
    hq, hkv = rng.choice(HEADS)
    if op in ("attend", "scores"):
        # At most 131,072 tokens in one cache, and as many bytes as the largest listed case.
        most = min(131072, (131072 if layout in ("default", "fast") else 16384) * 8 // max(hkv, 8))
        batch = rng.choice([1, 1, 1, 2, 4, 7, 16])
        tokens = _log_uniform(rng, 70, max(140, most // batch))
        if op == "scores":
            tokens = max(PAGE, tokens // 4 // PAGE * PAGE)
        return {"op": op, "layout": layout, "batch": batch, "hq": hq, "hkv": hkv, "tokens": tokens}
    if op == "prefill":
        dtype = rng.choice(["float16", "float16", "float32"])
        slow = dtype == "float32" or layout not in ("default", "fast")
        tokens = _log_uniform(rng, 64, (6100 if slow else 32773) * 8 // max(hkv, 8))
        return {"op": op, "layout": layout, "batch": 1, "hkv": hkv, "tokens": tokens, "dtype": dtype}
    if op == "fetch":
        tokens = _log_uniform(rng, 200, 8100 * 8 // max(hkv, 8))
        return {"op": op, "layout": layout, "batch": 1, "hkv": hkv, "tokens": tokens,
                "chunk": max(64, tokens // rng.randint(1, 4))}
    if op == "generate":
        return {"op": op, "layout": layout, "batch": 1, "hq": hq, "hkv": hkv, "tokens": rng.randint(20, 1000),
                "steps": rng.randint(10, 40)}
    tokens = _log_uniform(rng, 64, 8192 * 8 // max(hkv, 8)) // PAGE * PAGE
    return {"op": op, "layout": layout if layout in ("default", "fast") else "default", "batch": 1, "hq": hq,
            "hkv": hkv, "tokens": max(PAGE, tokens)}


# ---- inputs ---------------------------------------------------------------------


def _config(case):
    int8, l1, deep, split = LAYOUTS[case["layout"]]
    return TurboPolarConfig(num_q_heads=case.get("hq", case["hkv"]), num_kv_heads=case["hkv"], use_int8_radii=int8,
                            k_angle_bits_level1=l1, k_angle_bits_deep=deep, split_dim=split)


def _inputs(case, seed):
    """Keys with per-channel scales, as a model's keys have them, values and queries."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    dtype = getattr(torch, case.get("dtype", "float16"))
    total = case["tokens"] + case.get("steps", 0)
    shape = (case["batch"], case["hkv"], total, DIM)
    channel = torch.exp((torch.rand((1, case["hkv"], 1, DIM), generator=g, device="cuda") * 2 - 1) * math.log(4.0))
    k = (torch.randn(shape, generator=g, device="cuda") * channel).to(dtype)
    v = torch.randn(shape, generator=g, device="cuda").to(dtype)
    q = torch.randn((max(1, case.get("steps", 0)), case["batch"], case.get("hq", case["hkv"]), DIM), generator=g,
                    device="cuda").to(torch.float16)
    return k, v, q


def _residuals(case, seed):
    """Residuals of the size that the key quantiser leaves."""
    g = torch.Generator(device="cuda").manual_seed(int(seed) + 1)
    shape = (case["batch"], case["hkv"], case["tokens"] // PAGE, PAGE, DIM)
    return (torch.randn(shape, generator=g, device="cuda") * 0.05).to(torch.float16)


def prepare(case, seed):
    k, v, q = _inputs(case, seed)
    cfg = _config(case)
    op = case["op"]
    state = {"case": case, "cfg": cfg}
    if op in ("attend", "scores", "qjl"):
        # The cache that the prompt and the tokens so far have filled.
        cache = TurboPolarKVCacheRuntime(cfg)
        cache.append(k, v)
        state.update(cache=cache, bridge=HipKernelBridge(), q=q[0])
        if op == "qjl":
            sketcher = QJLResidualEncoder(cfg)
            sketcher.W("cuda")
            state.update(sketcher=sketcher, residuals=_residuals(case, seed))
    elif op == "prefill":
        state.update(k=k, v=v)
    elif op == "fetch":
        step = case["chunk"]
        cuts = range(0, case["tokens"], step)
        state.update(chunks=[(k[:, :, c:c + step].contiguous(), v[:, :, c:c + step].contiguous()) for c in cuts])
    else:
        n = case["tokens"]
        state.update(prompt=(k[:, :, :n].contiguous(), v[:, :, :n].contiguous()), steps=[
            (q[i][:, :, None], k[:, :, n + i:n + i + 1].contiguous(), v[:, :, n + i:n + i + 1].contiguous())
            for i in range(case["steps"])])
    return state


# ---- one pass -------------------------------------------------------------------


def _full(*tensors):
    return [t for t in tensors if t is not None and t.numel()]


def run(state):
    op, cfg = state["case"]["op"], state["cfg"]
    if op == "attend":
        block, quant_v, tail_k, tail_v, _, length = state["cache"].get_fused_attention_inputs()
        if tail_k is None:
            return state["bridge"].execute_online_attention_quant_v(state["q"], block, quant_v, None, None, cfg,
                                                                    length)[0]
        return state["bridge"].execute_online_attention_quant_v_dense_tail(
            state["q"], block, quant_v, tail_k, tail_v, None, None, cfg, length)[0]
    if op == "scores":
        block = state["cache"].get_fused_attention_inputs()[0]
        return state["bridge"].execute_fused_qk(state["q"], block, cfg)
    if op == "qjl":
        block, quant_v, _, _, _, length = state["cache"].get_fused_attention_inputs()
        payload = state["sketcher"].compute_residual_sketch(state["residuals"])
        signs = state["sketcher"].query_signs(state["q"])
        out, _ = state["bridge"].execute_online_attention_quant_v(state["q"], block, quant_v, payload, signs, cfg,
                                                                  length, use_qjl=True)
        return {"attention": out, "norms": payload.norms, "signs": payload.packed_signs, "query_signs": signs}
    if op == "prefill":
        cache = TurboPolarKVCacheRuntime(cfg)
        cache.append(state["k"], state["v"])
        block, quant_v, tail_k, tail_v, _, _ = cache.get_fused_attention_inputs()
        pages = [] if block is None else _full(block.radii, block.angle_codes_l1, block.angle_codes_deep,
                                               block.radii_scales, quant_v.codes, quant_v.scales)
        return pages + _full(tail_k, tail_v)
    cache = TurboPolarFastCache(cfg)
    if op == "fetch":
        for k, v in state["chunks"]:
            keys, values = cache.update_and_fetch(k, v)
        return {"keys": keys, "values": values}
    cache.update_and_fetch(*state["prompt"])
    return [cache.decode_attention(q, k, v, cfg.attention_scale) for q, k, v in state["steps"]]


# ---- what a pass cannot do without ------------------------------------------------


def _token_bytes(case):
    """Compressed bytes of one token of one kv head: (key, value)."""
    int8, l1, deep, split = LAYOUTS[case["layout"]]
    key = PAIRS * (1 if int8 else 2) + -(-(split // 2) * l1 // 8) + -(-(PAIRS - split // 2) * deep // 8)
    return key + (2 / PAGE if int8 else 0), DIM + DIM // 32 * 2


def work(case):
    rows, tokens = case["batch"] * case["hkv"], case["tokens"]
    key, value = _token_bytes(case)
    item = 4 if case.get("dtype") == "float32" else 2
    heads = case["batch"] * case.get("hq", case["hkv"])
    pages = tokens // PAGE * PAGE
    tail = tokens - pages
    dense = 2 * DIM * item
    op = case["op"]
    if op == "attend":
        return {"bytes": rows * (pages * (key + value) + tail * 512) + heads * 512, "flops": 4 * heads * tokens * DIM}
    if op == "scores":
        return {"bytes": rows * pages * key + heads * (256 + 2 * pages), "flops": 2 * heads * pages * DIM}
    if op == "prefill":
        return {"bytes": rows * (tokens * dense + pages * (key + value) + tail * dense), "flops": 30 * rows * tokens * DIM}
    if op == "fetch":
        done, moved = 0, 0
        while done < tokens:
            n = min(case["chunk"], tokens - done)
            done += n
            # the chunk in, its pages out, the whole history back
            moved += n * (dense + key + value) + done * (key + value + 512)
        return {"bytes": rows * moved, "flops": 30 * rows * tokens * DIM}
    if op == "generate":
        bytes_ = rows * tokens * (dense + 2 * (key + value) + 512)
        flops = 0
        for i in range(case["steps"]):
            n = tokens + i + 1
            full = n // PAGE * PAGE
            bytes_ += rows * (2 * dense + full * (key + value) + (n - full) * 512) + heads * 512
            flops += 4 * heads * n * DIM
        return {"bytes": bytes_, "flops": flops}
    bits = 64
    return {"bytes": rows * tokens * (256 + 2 * (bits // 8 + 2) + key + value) + DIM * bits * 4 + heads * 520,
            "flops": 2 * rows * tokens * DIM * bits + 4 * heads * tokens * DIM}


def tolerance(case):
    op = case["op"]
    if op == "prefill":
        # Codes are whole numbers, and radii and scales are correctly rounded fp16.
        return "exact"
    if op == "fetch":
        # One fp16 rounding of the product of two fp32 functions.
        return {"rel": 8e-4, "max": 4e-3}
    if op == "scores":
        return {"rel": 2e-3, "max": 2e-2}
    # fp16 weights, fp16 keys and values in the products, fp32 sums, an fp16
    # result; sketch bits may differ where a projection is a rounding from zero.
    return {"rel": 2e-3, "max": 2e-2, "differ": 1e-5}


# ---- the same in 64 bits ------------------------------------------------------------


def _encode(k, layout):
    """Whole pages of keys ``[..., 64, 128]`` as (radii, log scale, codes): the fp16
    (or fp32) operation sequence of the format, each step rounded once."""
    int8, l1, deep, split = LAYOUTS[layout]
    half = k.dtype == torch.float16
    x, y = k[..., 0::2].double(), k[..., 1::2].double()
    if half:
        square = (x * x).half().double() + (y * y).half().double()
        radii = square.half().double().sqrt().half()
        angle = torch.atan2(y, x).half().double()
        turn = ((angle + 3.140625).half().double() / 6.28125).half().double().clamp(0, 1)
    else:
        radii = (x.float() * x.float() + y.float() * y.float()).sqrt().half()
        turn = ((torch.atan2(y, x).float() + math.pi) / (2 * math.pi)).clamp(0, 1)
        turn = torch.where(turn > 1 - 1e-6, torch.zeros_like(turn), turn).double()
    levels = torch.full((PAIRS,), float(2 ** deep - 1), dtype=torch.float64, device=k.device)
    levels[: split // 2] = float(2 ** l1 - 1)
    codes = (turn.float() * levels.float()).round()
    scale = None
    if int8:
        log = radii.clamp(min=torch.tensor(1e-6).half().item()).double().log().half().double()
        top = log.abs().amax(dim=(-2, -1), keepdim=True)
        scale = (torch.where(top == 0, torch.full_like(top, 1e-6), top).float() / 127).half().double()
        radii = (log / scale).float().round().clamp(-128, 127)
    return radii, scale, codes, levels


def _keys64(k, layout):
    """Decoded keys of ``[B, H, T, 128]`` inputs, T whole pages."""
    B, H, T, _ = k.shape
    radii, scale, codes, levels = _encode(k.reshape(B, H, T // PAGE, PAGE, DIM), layout)
    r = radii.double() if scale is None else torch.exp(radii.double() * scale)
    angle = codes.double() / levels * (2 * math.pi) - math.pi
    return torch.stack((r * torch.cos(angle), r * torch.sin(angle)), dim=-1).reshape(B, H, T, DIM)


def _values64(v):
    B, H, T, _ = v.shape
    x = v.reshape(B, H, T, 4, 32).double()
    s = (x.abs().amax(dim=-1, keepdim=True).float() / 127).half()
    s = torch.where(s == 0, torch.full_like(s, 1e-4), s).double()
    q = x / s if v.dtype == torch.float32 else (x / s).half().double()
    return (q.round().clamp(-128, 127) * s).reshape(B, H, T, DIM)


def _scale64():
    return float(torch.tensor(1.0 / math.sqrt(DIM)).half())


def _attend64(q, keys, values, extra=None):
    """``q`` [B, Hq, 128] over ``keys`` / ``values`` [B, H, T, 128]; ``extra`` adds to the dot products."""
    B, H, T, _ = keys.shape
    q = q.double().reshape(B, H, -1, DIM)
    out = torch.empty_like(q)
    for b in range(B):
        for h in range(H):
            s = q[b, h] @ keys[b, h].T
            if extra is not None:
                s = s + extra[b, h]
            out[b, h] = torch.softmax(s * _scale64(), dim=-1) @ values[b, h]
    return out.reshape(B, -1, DIM)


def _history64(k, v, layout, tokens):
    full = tokens // PAGE * PAGE
    keys = torch.cat((_keys64(k[:, :, :full], layout), k[:, :, full:tokens].double()), dim=2)
    values = torch.cat((_values64(v[:, :, :full]), v[:, :, full:tokens].double()), dim=2)
    return keys, values


def exact(case, seed):
    op, layout, tokens = case["op"], case["layout"], case["tokens"]
    k, v, q = _inputs(case, seed)
    if op == "attend":
        out = torch.empty_like(q[0], dtype=torch.float64)
        g = case["hq"] // case["hkv"]
        for h in range(case["hkv"]):  # one kv head at a time, for memory
            keys, values = _history64(k[:, h:h + 1], v[:, h:h + 1], layout, tokens)
            out[:, h * g:(h + 1) * g] = _attend64(q[0][:, h * g:(h + 1) * g], keys, values)
        return out
    if op == "scores":
        g = case["hq"] // case["hkv"]
        out = torch.empty((case["batch"], case["hq"], tokens), dtype=torch.float64, device="cuda")
        for h in range(case["hkv"]):
            keys = _keys64(k[:, h:h + 1], layout)[:, 0]
            for b in range(case["batch"]):
                out[b, h * g:(h + 1) * g] = q[0][b, h * g:(h + 1) * g].double() @ keys[b].T * _scale64()
        return out
    if op == "qjl":
        bits = 64
        e = _residuals(case, seed)
        w = torch.from_numpy(qjl_projection(42, DIM, bits)).cuda().double()
        mine = torch.where(e.reshape(case["batch"], case["hkv"], tokens, DIM).double() @ w >= 0, 1.0, -1.0)
        theirs = torch.where(q[0].double() @ w >= 0, 1.0, -1.0)
        norms = e.double().square().sum(-1).sqrt()
        qn = q[0].double().square().sum(-1).reshape(case["batch"], case["hkv"], -1, 1)
        theirs = theirs.reshape(case["batch"], case["hkv"], -1, bits)
        agree = theirs @ mine.transpose(2, 3) / bits  # (P - 2 hamming) / P
        rounded = norms.half().double().reshape(case["batch"], case["hkv"], 1, tokens)
        extra = rounded * qn.sqrt() * torch.sin(math.pi / 2 * agree)
        keys, values = _history64(k, v, layout, tokens)
        return {"attention": _attend64(q[0], keys, values, extra), "norms": norms, "signs": None, "query_signs": None}
    if op == "prefill":
        full = tokens // PAGE * PAGE
        B, H = case["batch"], case["hkv"]
        radii, scale, _, _ = _encode(k[:, :, :full].reshape(B, H, full // PAGE, PAGE, DIM), layout)
        int8, _, _, split = LAYOUTS[layout]
        x = v[:, :, :full].reshape(B, H, full // PAGE, PAGE, 4, 32).double()
        vs = x.abs().amax(dim=-1) / 127
        out = []
        if full:
            xk = k[:, :, :full].reshape(B, H, full // PAGE, PAGE, DIM).double()
            out = [None if int8 else (xk[..., 0::2].square() + xk[..., 1::2].square()).sqrt()]
            out += [None] * ((split > 0) + (split < DIM))
            out += ([scale] if int8 else []) + [None, vs]
        return out + _full(k[:, :, full:].double(), v[:, :, full:].double())
    if op == "fetch":
        pad = -tokens % PAGE
        k, v = (torch.nn.functional.pad(t, (0, 0, 0, pad)) for t in (k, v))
        return {"keys": _keys64(k, layout)[:, :, :tokens], "values": _values64(v)[:, :, :tokens]}
    full = [_history64(k, v, layout, (tokens + i + 1) // PAGE * PAGE) for i in range(case["steps"])]
    out = []
    for i in range(case["steps"]):
        keys, values = full[i]
        n, done = tokens + i + 1, keys.shape[2]
        out.append(_attend64(q[i], torch.cat((keys, k[:, :, done:n].double()), 2),
                             torch.cat((values, v[:, :, done:n].double()), 2)))
    return out
