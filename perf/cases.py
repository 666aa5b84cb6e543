"""The work this library is measured on: quantized matmuls of every weight
type the GGUF path takes, from one decode row to a prompt of hundreds, the
prompt's attention, and whole forwards of a Llama-shaped model.

Everything goes through the package's public entry points (QMatMul on device
buffers, the C ABI's attention call, Llama.forward and
Llama.decode_step_graph).  Weights are Gaussian values quantised here, block
by block, so that scales, minimums and quants have the distributions of real
files; activations are Gaussian with a spread of channel scales, as a norm's
output has.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import arm_ai_amd as A
from arm_ai_amd import _lib, llama

TYPES = {"q4_0": 2, "q5_0": 6, "q8_0": 8, "q2_k": 10, "q3_k": 11, "q4_k": 12, "q5_k": 13, "q6_k": 14}
BLOCK = {"q4_0": 32, "q5_0": 32, "q8_0": 32, "q2_k": 256, "q3_k": 256, "q4_k": 256, "q5_k": 256, "q6_k": 256}
BLOCK_BYTES = {"q4_0": 18, "q5_0": 22, "q8_0": 34, "q2_k": 84, "q3_k": 110, "q4_k": 144, "q5_k": 176, "q6_k": 210}
LARGEST_MATMUL = 14336 * 4096 * 512  # n * k * m of the largest listed matmul
LARGEST_WEIGHT = 14336 * 4096


def listed():
    return [
        # one token of an 8B model: the gate or up projection
        {"name": "decode_q4k", "kind": "matmul", "type": "q4_k", "n": 14336, "k": 4096, "m": 1},
        # one token of a 135M model: rows of 576 fall back to 32-element blocks; latency and launches only
        {"name": "decode_q5_0_small", "kind": "matmul", "type": "q5_0", "n": 1536, "k": 576, "m": 1},
        # several sequences decoded together
        {"name": "batch5_q5k", "kind": "matmul", "type": "q5_k", "n": 5632, "k": 2048, "m": 5},
        {"name": "batch8_q4k", "kind": "matmul", "type": "q4_k", "n": 4096, "k": 14336, "m": 8},
        # a chat turn's prompt of a few dozen tokens, a ragged count
        {"name": "short_prompt_q4k", "kind": "matmul", "type": "q4_k", "n": 5632, "k": 2048, "m": 37},
        # prompts of hundreds of tokens: an 8B model's gate or up projection, TinyLlama's ffn_down,
        # an all-Q8_0 file, a low-bit file
        {"name": "prompt_q4k", "kind": "matmul", "type": "q4_k", "n": 14336, "k": 4096, "m": 512},
        {"name": "prompt_q6k", "kind": "matmul", "type": "q6_k", "n": 2048, "k": 5632, "m": 512},
        {"name": "prompt_q8_0", "kind": "matmul", "type": "q8_0", "n": 4096, "k": 4096, "m": 333},
        {"name": "prompt_q3k", "kind": "matmul", "type": "q3_k", "n": 4096, "k": 4096, "m": 200},
        # the attention of a long prompt at an 8B model's heads
        {"name": "attn_prompt", "kind": "attn", "n_head": 32, "n_kv": 8, "head_dim": 128, "m": 2048, "index_pos": 0},
        # a whole prompt, and one generated token after it, of a TinyLlama-shaped model of four layers
        {"name": "model_prompt", "kind": "prompt", "model": "tinyllama", "layers": 4, "m": 512},
        {"name": "model_decode", "kind": "decode", "model": "tinyllama", "layers": 4, "pos": 600},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    pick = rng.random()
    if pick < 0.70:
        t = rng.choice(sorted(TYPES) + ["q4_k", "q4_k", "q6_k"])  # Q4_K_M files are the common ones
        b = BLOCK[t]
        m = _log_int(rng, 1, 640)
        n = _log_int(rng, 256, 16384)
        if rng.random() < 0.7:
            n = (n + 63) // 64 * 64
        k = max(2, int(round(_log_int(rng, 512, 14336) / b))) * b
        while n * k > LARGEST_WEIGHT or n * k * m > LARGEST_MATMUL:
            n = max(256, n // 2)
            m = max(1, m * 3 // 4)
        return {"kind": "matmul", "type": t, "n": n, "k": k, "m": m}
    if pick < 0.85:
        n_head, n_kv, hd = rng.choice([(32, 4, 64), (9, 3, 64), (32, 8, 128), (32, 32, 64)])
        m = _log_int(rng, 16, 2048)
        return {"kind": "attn", "n_head": n_head, "n_kv": n_kv, "head_dim": hd, "m": m,
                "index_pos": rng.choice([0, 0, rng.randrange(1, 1 + (2048 - m) // 2)]) if m < 2000 else 0}
    model, layers = rng.choice(["tinyllama", "smollm"]), rng.randrange(1, 5)
    if pick < 0.93:
        return {"kind": "prompt", "model": model, "layers": layers, "m": _log_int(rng, 9, 512)}
    return {"kind": "decode", "model": model, "layers": layers, "pos": _log_int(rng, 16, 620)}


# ---------------------------------------------------------------- weights
def _f16(x):
    return x.to(torch.float16)


def _bytes(x):
    """The bytes of the last dimension's elements."""
    return x.contiguous().view(torch.uint8)


def _safe(d):
    return torch.where(d == 0, torch.ones_like(d), d)


def _quantise(t, w):
    """GGUF blocks (uint8 [n, bytes per row]) of the f32 weight w [n, k], and a
    function giving the f64 values that those blocks stand for."""
    n, k = w.shape
    u8 = torch.uint8
    if t in ("q4_0", "q5_0", "q8_0"):
        x = w.view(n, -1, 32)
        amax, at = x.abs().max(-1, keepdim=True)
        if t == "q8_0":
            d, zero, top = _f16(amax / 127), 0, 127
        else:
            zero, top = (8, 15) if t == "q4_0" else (16, 31)
            d = _f16(x.gather(-1, at) / -zero)
        q = torch.round(x / _safe(d.float())) + zero
        q = q.clamp(-127 if t == "q8_0" else 0, top).to(torch.int32)
        if t == "q8_0":
            parts = [_bytes(d), _bytes(q.to(torch.int8))]
        else:
            qs = (q[..., :16] & 15) | ((q[..., 16:] & 15) << 4)
            parts = [_bytes(d), qs.to(u8)]
            if t == "q5_0":
                bit = ((q >> 4) & 1).view(n, -1, 4, 8) << torch.arange(8, device=w.device, dtype=torch.int32)
                parts.insert(1, bit.sum(-1).to(u8))
        return torch.cat(parts, -1).reshape(n, -1), lambda: (d.double() * (q - zero).double()).view(n, k)
    sub = 32 if t in ("q4_k", "q5_k") else 16
    x = w.view(n, -1, 256 // sub, sub)
    if t in ("q2_k", "q4_k", "q5_k"):  # scale and minimum of each sub-block
        steps, top = {"q2_k": (3, 15), "q4_k": (15, 63), "q5_k": (31, 63)}[t]
        lo = x.amin(-1).clamp(max=0)
        s = (x.amax(-1).clamp(min=0) - lo) / steps
        d, dmin = _f16(s.amax(-1, keepdim=True) / top), _f16(-lo.amin(-1, keepdim=True) / top)
        sc = torch.round(s / _safe(d.float())).clamp(0, top).to(torch.int32)
        mn = torch.round(-lo / _safe(dmin.float())).clamp(0, top).to(torch.int32)
        q = torch.round((x + (dmin.float() * mn)[..., None]) / _safe(d.float() * sc)[..., None]).clamp(0, steps).to(torch.int32)
        value = lambda: ((d.double() * sc)[..., None] * q - (dmin.double() * mn)[..., None]).view(n, k)  # noqa: E731
        if t == "q2_k":
            qq = q.view(n, -1, 2, 4, 32)
            qs = qq[..., 0, :] | (qq[..., 1, :] << 2) | (qq[..., 2, :] << 4) | (qq[..., 3, :] << 6)
            parts = [(sc | (mn << 4)).to(u8), qs.to(u8).view(n, -1, 64), _bytes(d), _bytes(dmin)]
        else:
            packed = torch.cat([sc[..., :4] | ((sc[..., 4:] >> 4) << 6), mn[..., :4] | ((mn[..., 4:] >> 4) << 6),
                                (sc[..., 4:] & 15) | ((mn[..., 4:] & 15) << 4)], -1).to(u8)
            qq = q.view(n, -1, 4, 2, 32)
            qs = ((qq[..., 0, :] & 15) | ((qq[..., 1, :] & 15) << 4)).to(u8).view(n, -1, 128)
            parts = [_bytes(d), _bytes(dmin), packed, qs]
            if t == "q5_k":
                high = ((q >> 4) & 1) << torch.arange(8, device=w.device, dtype=torch.int32)[:, None]
                parts.insert(3, high.sum(-2).to(u8))
        return torch.cat(parts, -1).reshape(n, -1), value
    half, top = (4, 32) if t == "q3_k" else (32, 128)  # signed scales of 16 elements, no minimum
    amax, at = x.abs().max(-1, keepdim=True)
    s = (x.gather(-1, at) / -half).squeeze(-1)
    smax, at = s.abs().max(-1, keepdim=True)
    d = _f16(s.gather(-1, at) / -top)
    sc = torch.round(s / _safe(d.float())).clamp(-top, top - 1).to(torch.int32)
    q = torch.round(x / _safe(d.float() * sc)[..., None]).clamp(-half, half - 1).to(torch.int32)
    value = lambda: ((d.double() * sc)[..., None] * q).view(n, k)  # noqa: E731
    if t == "q6_k":
        g = (q + 32).view(n, -1, 2, 4, 32)
        ql = torch.stack([(g[..., 0, :] & 15) | ((g[..., 2, :] & 15) << 4), (g[..., 1, :] & 15) | ((g[..., 3, :] & 15) << 4)], -2)
        qh = (g[..., 0, :] >> 4) | ((g[..., 1, :] >> 4) << 2) | ((g[..., 2, :] >> 4) << 4) | ((g[..., 3, :] >> 4) << 6)
        parts = [ql.to(u8).reshape(n, -1, 128), qh.to(u8).reshape(n, -1, 64), _bytes(sc.to(torch.int8)), _bytes(d)]
    else:
        g = (q + 4).view(n, -1, 2, 4, 32)
        bit = torch.arange(8, device=w.device, dtype=torch.int32).view(2, 4, 1)
        hmask = ((g >> 2) << bit).sum((-3, -2))
        qs = ((g & 3) << (2 * torch.arange(4, device=w.device, dtype=torch.int32).view(4, 1))).sum(-2)
        s6 = sc + 32
        packed = torch.cat([(s6[..., 0:4] & 15) | ((s6[..., 8:12] & 15) << 4), (s6[..., 4:8] & 15) | ((s6[..., 12:16] & 15) << 4),
                            (s6[..., 0:4] >> 4) | ((s6[..., 4:8] >> 4) << 2) | ((s6[..., 8:12] >> 4) << 4) | ((s6[..., 12:16] >> 4) << 6)], -1)
        parts = [hmask.to(u8), qs.to(u8).reshape(n, -1, 64), packed.to(u8), _bytes(d)]
    return torch.cat(parts, -1).reshape(n, -1), value


# ---------------------------------------------------------------- inputs
_ctx = None


def _context():
    """The process's library context: one device, one stream, as a program keeps it."""
    global _ctx
    if _ctx is None:
        torch.cuda.init()
        _ctx = A.Context(0)
    return _ctx


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _normal(g, *shape):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)


def _matmul_inputs(case, seed):
    g = _generator(seed)
    blocks, value = _quantise(case["type"], _normal(g, case["n"], case["k"]) / math.sqrt(case["k"]))
    x = _normal(g, case["m"], case["k"]) * torch.exp(0.4 * _normal(g, case["k"]))
    return blocks, value, x


def _attn_inputs(case, seed):
    g = _generator(seed)
    m, pos, hd = case["m"], case["index_pos"], case["head_dim"]
    qk = _normal(g, m, (case["n_head"] + case["n_kv"]) * hd)  # wq|wk's output
    v = _normal(g, m, case["n_kv"] * hd)
    max_seq = (pos + m + 511) // 512 * 512
    kc, vc = torch.zeros((2, case["n_kv"], max_seq, hd), device="cuda")
    kc[:, :pos] = _normal(g, case["n_kv"], pos, hd)
    vc[:, :pos] = _normal(g, case["n_kv"], pos, hd)
    theta = 1.0 / 10000.0 ** (torch.arange(0, hd, 2, dtype=torch.float64, device="cuda") / hd)
    angle = torch.arange(max_seq, dtype=torch.float64, device="cuda")[:, None] * theta
    return qk, v, torch.cos(angle).float(), torch.sin(angle).float(), kc, vc


def _config(case, max_seq):
    if case["model"] == "smollm":
        cfg = llama.smollm_135m_config(max_seq)
        cfg.n_layer = case["layers"]
        return cfg, llama.fallback_q4km_types, "q8_0"
    return llama.LlamaConfig(n_layer=case["layers"], max_seq=max_seq), llama.tinyllama_q4km_types, "q6_k"


def _model(case, seed):
    """A model of the named architecture with weights made from the seed."""
    cfg, types, head = _config(case, 640)
    names = {v: k for k, v in TYPES.items()}
    g = _generator(seed)

    def tensor(t, n, k):
        blocks, _ = _quantise(t, _normal(g, n, k) / math.sqrt(k))
        return A.QTensor(TYPES[t], (n, k), blocks.cpu().numpy())

    hw = llama.HostWeights(cfg)
    for layer in range(cfg.n_layer):
        t = types(cfg, layer)
        hw.layers.append({name: tensor(names[t[name]], n, k) for name, (n, k) in llama.weight_shapes(cfg).items()})
        hw.attn_norm.append((1 + 0.05 * _normal(g, cfg.hidden)).cpu().numpy())
        hw.ffn_norm.append((1 + 0.05 * _normal(g, cfg.hidden)).cpu().numpy())
    hw.tok_embeddings = _normal(g, cfg.vocab, cfg.hidden).cpu().numpy()
    hw.norm = (1 + 0.05 * _normal(g, cfg.hidden)).cpu().numpy()
    hw.output = tensor(head, cfg.vocab, cfg.hidden)
    n = case["m"] if case["kind"] == "prompt" else case["pos"]
    return llama.Llama(_context(), hw), torch.randint(cfg.vocab, (n + 1,), generator=g, device="cuda")


def prepare(case, seed):
    ctx = _context()
    if case["kind"] == "matmul":
        blocks, _, x = _matmul_inputs(case, seed)
        torch.cuda.synchronize()  # the library reads the blocks on its own stream
        mm = A.QMatMul.from_device_blocks(ctx, TYPES[case["type"]], (case["n"], case["k"]), blocks.data_ptr(), blocks.numel())
        return {"case": case, "mm": mm, "x": x, "y": torch.empty((case["m"], case["n"]), device="cuda")}
    if case["kind"] == "attn":
        qk, v, cos, sin, kc, vc = _attn_inputs(case, seed)
        out = torch.empty((case["m"], case["n_head"] * case["head_dim"]), device="cuda")
        return {"case": case, "ctx": ctx, "qk": qk, "v": v, "cos": cos, "sin": sin, "kc": kc, "vc": vc, "out": out}
    model, tokens = _model(case, seed)
    if case["kind"] == "decode":
        model.forward(tokens[:-1], 0)
        token = int(tokens[-1])
        model.decode_step_graph(token, case["pos"])  # a program's first token captures the step
        return {"case": case, "model": model, "token": token}
    return {"case": case, "model": model, "tokens": tokens[:-1]}


def run(state):
    case = state["case"]
    if case["kind"] == "matmul":
        state["mm"].forward_device(state["x"].data_ptr(), case["m"], state["y"].data_ptr())
        return state["y"]
    if case["kind"] == "attn":
        qk, v, h, hd = state["qk"], state["v"], case["n_head"], case["head_dim"]
        _lib.check(_lib.load().aq_llama_attn_prefill(
            state["ctx"].handle, qk.data_ptr(), qk.stride(0), qk.data_ptr() + 4 * h * hd, qk.stride(0), v.data_ptr(), v.stride(0),
            state["cos"].data_ptr(), state["sin"].data_ptr(), case["index_pos"], case["m"], state["kc"].data_ptr(),
            state["vc"].data_ptr(), h, case["n_kv"], hd, state["kc"].shape[1], state["out"].data_ptr()))
        return {"out": state["out"], "k": state["kc"], "v": state["vc"]}
    model = state["model"]
    logits = model.forward(state["tokens"], 0) if case["kind"] == "prompt" else model.decode_step_graph(state["token"], case["pos"])
    return {"logits": logits, "k": model.k_cache, "v": model.v_cache}


def work(case):
    if case["kind"] == "matmul":
        n, k, m = case["n"], case["k"], case["m"]
        return {"bytes": n * k // BLOCK[case["type"]] * BLOCK_BYTES[case["type"]] + 4 * m * (n + k), "flops": 2 * m * n * k}
    if case["kind"] == "attn":
        h, kv, hd, m, pos = (case[c] for c in ("n_head", "n_kv", "head_dim", "m", "index_pos"))
        keys = m * pos + m * (m + 1) // 2  # (query, key) pairs of one head
        return {"bytes": 4 * hd * (2 * m * h + 4 * m * kv + 2 * pos * kv), "flops": 4 * hd * h * keys}
    cfg, types, head = _config(case, 640)
    names = {v: k for k, v in TYPES.items()}
    m = case["m"] if case["kind"] == "prompt" else 1
    pos = 0 if case["kind"] == "prompt" else case["pos"]
    total = cfg.vocab * cfg.hidden // BLOCK[head] * BLOCK_BYTES[head] + 4 * (m * cfg.hidden + cfg.vocab)
    flops = 2 * cfg.vocab * cfg.hidden
    for layer in range(cfg.n_layer):
        t = types(cfg, layer)
        for name, (n, k) in llama.weight_shapes(cfg).items():
            total += n * k // BLOCK[names[t[name]]] * BLOCK_BYTES[names[t[name]]]
            flops += 2 * m * n * k
        total += 8 * cfg.head_dim * cfg.n_kv_head * (m + pos)
        flops += 4 * cfg.head_dim * cfg.n_head * (m * pos + m * (m + 1) // 2)
    return {"bytes": total, "flops": flops}


def tolerance(case):
    if case["kind"] == "matmul":  # exact integer block sums, f32 sums over the blocks
        return {"rel": 2e-6}
    if case["kind"] == "attn":  # f32 scores, softmax and sums
        return {"rel": 4e-6}
    # A value that another order of f32 sums moves across a rounding boundary
    # of the 8-bit activation quantiser moves by a whole quant, and what
    # follows with it: a few quantisers on, the difference is the rounding
    # error of 8 bits itself.  One prompt fed whole and in two pieces (other
    # tiles and K splits, the same model) differs by 0.017 in four layers.
    return {"rel": 0.03, "max": 0.3}


# ---------------------------------------------------------------- 64 bits
def _round_away(v):
    return np.sign(v) * np.floor(np.abs(v).astype(np.float64) + 0.5)


def _activation(x, q8k):
    """The f64 values that the activation's quantised blocks stand for: the
    format's own f32 arithmetic (Q8_K: 256 elements, d = 1 / (-128 / max);
    Q8_0: 32 elements, d = max / 127 rounded to f16)."""
    m, k = x.shape
    b = x.cpu().numpy().reshape(m, -1, 256 if q8k else 32)
    one = np.float32(1)
    if q8k:
        top = np.take_along_axis(b, np.abs(b).argmax(-1)[..., None], -1)
        scale = np.float32(-128) / top
        q = np.minimum(_round_away(scale * b), 127)
        d = (one / scale).astype(np.float64)
    else:
        d = np.abs(b).max(-1, keepdims=True) / np.float32(127)
        q = _round_away(b * (one / d))
        d = d.astype(np.float16).astype(np.float64)
    return torch.from_numpy((d * q).reshape(m, k)).cuda()


def exact(case, seed):
    if case["kind"] == "matmul":
        _, value, x = _matmul_inputs(case, seed)
        return _activation(x, BLOCK[case["type"]] == 256) @ value().T
    if case["kind"] == "attn":
        qk, v, cos, sin, kc, vc = (t.double() for t in _attn_inputs(case, seed))
        h, kv, hd, m, pos = (case[c] for c in ("n_head", "n_kv", "head_dim", "m", "index_pos"))
        c, s = cos[pos:pos + m, None], sin[pos:pos + m, None]

        def rotate(t):
            a, b = t[..., 0::2], t[..., 1::2]
            return torch.stack([a * c - b * s, a * s + b * c], -1).flatten(-2)

        q = rotate(qk[:, :h * hd].view(m, h, hd))
        kc[:, pos:pos + m] = rotate(qk[:, h * hd:].view(m, kv, hd)).transpose(0, 1)
        vc[:, pos:pos + m] = v.view(m, kv, hd).transpose(0, 1)
        hidden = torch.ones((m, pos + m), dtype=torch.bool, device="cuda").triu(pos + 1)
        out = torch.empty((m, h, hd), dtype=torch.float64, device="cuda")
        for i in range(h):
            score = q[:, i].contiguous() @ kc[i * kv // h, :pos + m].T.contiguous() / math.sqrt(hd)
            out[:, i] = score.masked_fill(hidden, -math.inf).softmax(-1) @ vc[i * kv // h, :pos + m]
        return {"out": out.view(m, h * hd), "k": kc, "v": vc}
    # Whole models have no such value: the 8-bit rounding of every layer's
    # activations makes a step of a quant out of an error in the last bit,
    # or none, by chance.
    return None
