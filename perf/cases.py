"""Performance cases of the attention path: what users of this package have it do, through its
public entry points, from calls bound by latency to calls that fill the GPU.

Kinds of case (`case["kind"]`):
  sdpa     F.scaled_dot_product_attention without gradients: prompts (many query rows) and decode
           steps (one query row), dense or GGUF Q8_0 keys and values
  train    the same forward with autograd, and its backward
  cache    a generation session on a KVCache: clear, append the prompt with RoPE, attend to it, then
           decode steps of one token (append, attend)
  mha      nn.MultiheadAttention as its defaults run it (averaged weights returned), forward and backward

`listed()` names one case per way of use; `draw()` varies the sizes, data types and options of each
over the range that its listed case stands for.
"""

from __future__ import annotations

import math
import random

import torch

from gguf_train_amd import KVCache, QuantizedTensor
from gguf_train_amd.nn import MultiheadAttention
from gguf_train_amd.nn import functional as F

DEV = "cuda"
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
SIZE = {"fp16": 2, "bf16": 2, "fp32": 4, "q8_0": 34 / 32}


def _case(name, kind, role, dtype, B, H, Hkv, L, S, D, causal=False, mask="none", kv="dense", dropout=0.0, steps=0):
    return {"name": name, "kind": kind, "role": role, "dtype": dtype, "B": B, "H": H, "Hkv": Hkv, "L": L, "S": S, "D": D,
            "causal": causal, "mask": mask, "kv": kv, "dropout": dropout, "steps": steps}


def listed():
    return [
        # a small call in the default dtype: a test, a toy model, one layer of a tiny one; latency is all of it
        _case("small_fp32", "sdpa", "small", "fp32", 1, 4, 4, 128, 128, 64, causal=True),
        # the prompt of a batch of sequences, multi-head, fp16
        _case("prompt_fp16", "sdpa", "prompt", "fp16", 4, 32, 32, 2048, 2048, 128, causal=True),
        # one long prompt of an odd length, grouped-query, bf16 (most models' dtype)
        _case("prompt_bf16_gqa_long", "sdpa", "prompt", "bf16", 1, 32, 8, 4001, 4001, 128, causal=True),
        # a chunk of a prompt over the keys that came before it: is_causal is aligned to the top left, so
        # such a caller passes the causal band as a mask, in the queries' dtype or as bool
        _case("chunk_masked_fp16", "sdpa", "chunk", "fp16", 4, 32, 8, 500, 1500, 128, mask="band"),
        # one decode step of a serving batch, grouped-query, fp16 keys and values
        _case("decode_fp16", "sdpa", "decode", "fp16", 32, 32, 8, 1, 4096, 128),
        # the same over GGUF Q8_0 keys and values, fp16 queries
        _case("decode_q8_fp16", "sdpa", "decode_q8", "fp16", 16, 32, 8, 1, 8192, 128, kv="q8_0"),
        # and for a bf16 model, a smaller batch, an odd length
        _case("decode_q8_bf16", "sdpa", "decode_q8", "bf16", 4, 32, 8, 1, 3001, 128, kv="q8_0"),
        # a generation session on a Q8_0 cache: prompt, then decode steps; launches and host work count
        _case("session_q8", "cache", "session", "fp16", 4, 32, 8, 500, 500, 128, causal=True, kv="q8_0", steps=8),
        # one layer's attention of a training step, padded batch, bf16
        _case("train_bf16", "train", "train", "bf16", 8, 16, 16, 1024, 1024, 64, causal=True, mask="pad"),
        # the same with dropout of the probabilities, a ragged length
        _case("train_bf16_dropout", "train", "train", "bf16", 4, 16, 16, 777, 777, 64, causal=True, mask="pad", dropout=0.1),
        # a head size that is no power of two
        _case("train_fp16_head80", "train", "train", "fp16", 4, 16, 16, 1000, 1000, 80, causal=True),
        # a self-attention layer in the default dtype with its default arguments, padded batch
        _case("mha_fp32", "mha", "mha", "fp32", 8, 8, 8, 256, 256, 64, mask="pad"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    role = rng.choice(["small", "prompt", "prompt", "chunk", "decode", "decode_q8", "decode_q8", "session", "train", "train",
                       "mha"])
    half = rng.choice(["fp16", "bf16"])
    if role == "small":
        return _trim(_case("", "sdpa", role, rng.choice(["fp32", "fp16", "bf16"]), rng.randint(1, 2), rng.choice([2, 4, 8]), 2,
                           _log(rng, 16, 256), 0, rng.choice([64, 128]), causal=rng.random() < 0.7))
    if role == "prompt":
        H = rng.choice([8, 16, 32])
        Hkv = H // rng.choice([1, 2, 4])
        L, D = _log(rng, 128, 4096), rng.choice([64, 128, 128])
        # batch: up to what the listed prompts cost
        most = int(131e9 / (2.0 * D * H * L * (L + 1)))
        return _trim(_case("", "sdpa", role, half, _log(rng, 1, max(1, min(16, most))), H, Hkv, L, 0, D, causal=True))
    if role == "chunk":
        H = rng.choice([8, 16, 32])
        L = _log(rng, 32, 512)
        return _trim(_case("", "sdpa", role, half, rng.randint(1, 4), H, H // rng.choice([1, 4]), L, L + _log(rng, 32, 1024),
                           rng.choice([64, 128]), mask=rng.choice(["band", "band_bool"])))
    if role in ("decode", "decode_q8"):
        q8 = role == "decode_q8"
        dtype = rng.choice(["fp16", "bf16"]) if not q8 else rng.choice(["fp16", "bf16", "fp32"])
        Hkv = rng.choice([4, 8])
        H = Hkv * rng.choice([1, 4, 8])
        S = _log(rng, 128, 8192)
        # fp16 batches up to the listed ones' bytes; other queries over Q8_0 up to the smaller listed one's
        rows = 32 * 4096 if not q8 else 16 * 8192 if dtype == "fp16" else 4 * 3001
        if q8 and dtype != "fp16":
            S, H = min(S, rows), min(H, 32)
        most = max(1, min(32, rows // S))
        return _trim(_case("", "sdpa", role, dtype, _log(rng, 1, most), H, Hkv, 1, S, rng.choice([64, 128]) if not q8 else 128,
                           mask=rng.choice(["none", "none", "pad"]), kv="q8_0" if q8 else "dense"))
    if role == "session":
        kv = rng.choice(["q8_0", "dense"])
        dtype = "fp16" if kv == "q8_0" else half
        Hkv = rng.choice([2, 4, 8])
        return _trim(_case("", "cache", role, dtype, rng.randint(1, 4), Hkv * rng.choice([1, 4]), Hkv, _log(rng, 20, 500), 0,
                           rng.choice([64, 128]), causal=True, kv=kv, steps=rng.randint(2, 8)))
    if role == "train":
        H = rng.choice([4, 8, 16])
        D = rng.choice([64, 64, 80, 96, 128])
        L = _log(rng, 64, 1024)
        B = _log(rng, 1, max(1, min(8, 4 * 16 * 1024 * (2 if D == 64 else 1) // (H * L))))
        return _trim(_case("", "train", role, half, B, H, H if D != 128 else H // rng.choice([1, 2]), L, 0, D, causal=True,
                           mask=rng.choice(["none", "pad"]), dropout=rng.choice([0.0, 0.0, 0.1])))
    H = rng.choice([4, 8])
    return _trim(_case("", "mha", role, "fp32", _log(rng, 1, 8), H, H, _log(rng, 16, 256), 0, 64, mask=rng.choice(["none", "pad"])))


def _trim(case):
    """Drawn cases carry no name; S = 0 stands for S = L, Hkv is a divisor of H."""
    del case["name"]
    if case["S"] == 0:
        case["S"] = case["L"]
    case["Hkv"] = max(1, math.gcd(case["H"], case["Hkv"]))
    return case


# ---- inputs ---------------------------------------------------------------------------------------


def _lengths(case, seed):
    """Key lengths of a padded batch: half to all of S."""
    r = random.Random(seed + 17)
    return [r.randint((case["S"] + 1) // 2, case["S"]) for _ in range(case["B"])]


def _normal(gen, shape, dtype, amp=1.0):
    return (amp * torch.randn(shape, generator=gen, device=DEV, dtype=torch.float32)).to(dtype)


def _q8_blocks(x):
    """GGUF Q8_0 blocks of x (last dimension a multiple of 32): scale amax / 127 as float16, quants
    rounded half away from zero."""
    b = x.float().reshape(-1, 32)
    d = b.abs().amax(1, keepdim=True) / 127.0
    inv = torch.where(d > 0, 1.0 / d, torch.zeros_like(d))
    y = b * inv
    qs = (torch.sign(y) * torch.floor(y.abs() + 0.5)).to(torch.int8)
    return torch.cat([d.half().view(torch.uint8).reshape(-1, 2), qs.view(torch.uint8)], 1).reshape(-1).contiguous()


def _q8_values(data, shape):
    b = data.reshape(-1, 34)
    d = b[:, :2].contiguous().view(torch.float16).double()
    return (d * b[:, 2:].contiguous().view(torch.int8).double()).reshape(shape)


def _mask(case, seed):
    """The mask as the caller passes it: key padding (B,1,1,S), or the (L,S) band of a chunk."""
    L, S = case["L"], case["S"]
    if case["mask"] == "none":
        return None
    if case["mask"] == "pad":
        keep = torch.arange(S, device=DEV)[None, :] < torch.tensor(_lengths(case, seed), device=DEV)[:, None]
        if case["kind"] == "mha":
            return ~keep  # torch.nn's convention: True is left out
        zero = torch.zeros((case["B"], 1, 1, S), dtype=torch.float32, device=DEV)
        return zero.masked_fill(~keep[:, None, None, :], float("-inf"))
    keep = torch.ones((L, S), dtype=torch.bool, device=DEV).tril(S - L)
    if case["mask"] == "band_bool":
        return keep
    return torch.zeros((L, S), dtype=DTYPES[case["dtype"]], device=DEV).masked_fill(~keep, float("-inf"))


def _tensors(case, seed):
    """q, k, v (and the output's gradient) of a seed; Q8_0 keys and values as their blocks."""
    gen = torch.Generator(device=DEV).manual_seed(seed)
    B, H, Hkv, L, S, D = (case[n] for n in ("B", "H", "Hkv", "L", "S", "D"))
    dt = DTYPES[case["dtype"]]
    if case["kind"] == "mha":
        E = H * D
        amp = 1.0 / math.sqrt(E)
        return {"x": _normal(gen, (B, L, E), dt), "w_in": _normal(gen, (3 * E, E), dt, amp), "b_in": _normal(gen, (3 * E,), dt, 0.1),
                "w_out": _normal(gen, (E, E), dt, amp), "b_out": _normal(gen, (E,), dt, 0.1), "dout": _normal(gen, (B, L, E), dt)}
    n = case["steps"]  # a session's tokens after the prompt
    t = {"q": _normal(gen, (B, H, L + n, D), dt), "k": _normal(gen, (B, Hkv, S + n, D), dt),
         "v": _normal(gen, (B, Hkv, S + n, D), dt)}
    if case["kind"] == "sdpa" and case["kv"] == "q8_0":
        for name in ("k", "v"):
            t[name] = _q8_blocks(t[name])
    if case["kind"] == "train":
        t["dout"] = _normal(gen, (B, H, L, D), dt)
    return t


def prepare(case, seed):
    t = _tensors(case, seed)
    state = {"case": case, "seed": seed, **t}
    shape = (case["B"], case["Hkv"], case["S"], case["D"])
    if case["kind"] in ("sdpa", "train"):
        state["mask"] = _mask(case, seed)
    if case["kind"] == "sdpa" and case["kv"] == "q8_0":
        state["k"], state["v"] = QuantizedTensor(t["k"], shape), QuantizedTensor(t["v"], shape)
    if case["kind"] == "train":
        for name in ("q", "k", "v"):
            state[name].requires_grad_(True)
    if case["kind"] == "cache":
        total = case["L"] + case["steps"]
        state["pos"] = torch.arange(total, device=DEV, dtype=torch.int32)
        state["cache"] = KVCache(case["B"], case["Hkv"], total, case["D"],
                                 "q8_0" if case["kv"] == "q8_0" else DTYPES[case["dtype"]], device=DEV)
    if case["kind"] == "mha":
        m = MultiheadAttention(case["H"] * case["D"], case["H"], batch_first=True, device=DEV, dtype=DTYPES[case["dtype"]])
        with torch.no_grad():
            m.in_proj_weight.copy_(t["w_in"])
            m.in_proj_bias.copy_(t["b_in"])
            m.out_proj.weight.copy_(t["w_out"])
            m.out_proj.bias.copy_(t["b_out"])
        state["module"] = m
        state["x"].requires_grad_(True)
        state["mask"] = _mask(case, seed)
    return state


# ---- one pass -------------------------------------------------------------------------------------

ROPE = {"mode": 2, "freq_base": 10000.0}


def run(state):
    case = state["case"]
    if case["kind"] == "sdpa":
        return F.scaled_dot_product_attention(state["q"], state["k"], state["v"], attn_mask=state["mask"],
                                              is_causal=case["causal"])
    if case["kind"] == "train":
        ins = (state["q"], state["k"], state["v"])
        if case["dropout"]:
            torch.default_generator.manual_seed(state["seed"])  # the same decisions on every pass
        out = F.scaled_dot_product_attention(*ins, attn_mask=state["mask"], dropout_p=case["dropout"], is_causal=case["causal"])
        return [out.detach(), *torch.autograd.grad(out, ins, state["dout"])]
    if case["kind"] == "cache":
        q, k, v, pos, cache, T = state["q"], state["k"], state["v"], state["pos"], state["cache"], case["L"]
        outs = []
        cache.clear()
        for lo, hi in [(0, T)] + [(i, i + 1) for i in range(T, T + case["steps"])]:
            cache.append(k[:, :, lo:hi], v[:, :, lo:hi], rope=ROPE)
            rq = F.rope(q[:, :, lo:hi], pos[lo:hi], mode=ROPE["mode"], freq_base=ROPE["freq_base"])
            outs.append(cache.attention(rq))
        return outs
    m, x = state["module"], state["x"]
    out, weights = m(x, x, x, key_padding_mask=state["mask"])
    ins = (x, m.in_proj_weight, m.in_proj_bias, m.out_proj.weight, m.out_proj.bias)
    return [out.detach(), weights, *torch.autograd.grad(out, ins, state["dout"])]


# ---- work -----------------------------------------------------------------------------------------


def _pairs(case):
    """(query, key) pairs of one head of one sequence that the masks leave (a padded sequence at its
    mean length, three quarters of S)."""
    L, S = case["L"], case["S"]
    if case["mask"].startswith("band"):
        return L * (S - L) + L * (L + 1) / 2
    v = 0.75 * S if case["mask"] == "pad" else S
    if case["causal"]:
        v = min(v, L)
        return v * (v + 1) / 2 + (L - v) * v
    return L * v


def work(case):
    B, H, Hkv, L, S, D, n = (case[x] for x in ("B", "H", "Hkv", "L", "S", "D", "steps"))
    es = SIZE[case["dtype"]]
    if case["kind"] == "cache":
        # rows in (dense), stored once, outputs; each step reads the keys and values held so far
        kvs = SIZE["q8_0"] if case["kv"] == "q8_0" else es
        T = L + n
        held = sum(range(L + 1, T + 1)) if n else 0
        rows = B * Hkv * D
        return {"bytes": int(2 * rows * T * (es + kvs) + 2 * B * H * T * D * es + 2 * rows * kvs * (held + L)),
                "flops": int(4 * D * B * H * (L * (L + 1) / 2 + held))}
    flops = 4 * D * B * H * _pairs(case)
    if case["kind"] == "mha":
        E = H * D
        return {"bytes": int(4 * (4 * B * L * E + B * L * S + 2 * (4 * E * E + 4 * E))),
                "flops": int(3.5 * flops + 3 * 8 * B * L * E * E)}
    q, kv = B * H * L * D, B * Hkv * S * D
    masked = {"none": 0, "pad": 4 * B * S, "band": es * L * S, "band_bool": L * S}[case["mask"]]
    if case["kind"] == "train":
        # q, k, v, dO in; O, dQ, dK, dV out
        return {"bytes": int(es * (4 * q + 4 * kv) + masked), "flops": int(3.5 * flops)}
    if case["mask"] == "pad":
        kv *= 0.75  # rows past a sequence's length need not be read
    kvs = SIZE["q8_0"] if case["kv"] == "q8_0" else es
    return {"bytes": int(2 * es * q + 2 * kvs * kv + masked), "flops": int(flops)}


# ---- expected results -----------------------------------------------------------------------------


def tolerance(case):
    # 2-norm of the difference over the result's, about four times the largest seen against exact()
    # (outputs are rounded to the inputs' dtype: float32 1.4e-6, float16 2.9e-4, bfloat16 1.7e-3;
    # a Q8_0 cache 4.9e-4, where a rotated key near a tie is quantized to the neighbouring value)
    if case["dtype"] == "fp32":
        return {"rel": 5e-6}
    if case["kind"] == "cache" and case["kv"] == "q8_0":
        return {"rel": 2e-3}
    return {"rel": 1.2e-3 if case["dtype"] == "fp16" else 7e-3}


def _attend64(q, k, v, bias):
    """float64 attention of one sequence: q (H,L,D), k, v (Hkv,S,D), bias (L,S) or (1,S); rows with
    nothing visible are 0.  Returns the output and the weights (H,L,S)."""
    g = q.shape[0] // k.shape[0]
    outs, ws = [], []
    for h in range(q.shape[0]):
        s = q[h] @ k[h // g].t().contiguous() / math.sqrt(q.shape[-1]) + bias
        p = torch.softmax(s, -1).nan_to_num(0.0)
        outs.append(p @ v[h // g])
        ws.append(p)
    return torch.stack(outs), ws


def _bias64(case, mask, b, L, S, device):
    bias = torch.zeros((L, S), dtype=torch.float64, device=device)
    if case["causal"]:
        bias.masked_fill_(~torch.ones((L, S), dtype=torch.bool, device=device).tril(), float("-inf"))
    if mask is not None:
        m = mask[b, 0] if mask.ndim == 4 else mask
        bias = bias.masked_fill(~m, float("-inf")) if m.dtype == torch.bool else bias + m.double()
    return bias


def _rope64(x, pos0):
    """NeoX rotation of x (..., T, D) at positions pos0 + t; the angles follow the float32 chain
    theta_{i+1} = theta_i * base^(-2/D) that the operator is defined by."""
    T, D = x.shape[-2:]
    step = torch.tensor(10000.0, dtype=torch.float32).pow(torch.tensor(-2.0 / D, dtype=torch.float32))
    theta = torch.arange(pos0, pos0 + T, dtype=torch.float32)
    cols = []
    for _ in range(D // 2):
        cols.append(theta)
        theta = theta * step
    ang = torch.stack(cols, 1).double().to(x.device)
    lo, hi = x[..., : D // 2].double(), x[..., D // 2:].double()
    c, s = ang.cos(), ang.sin()
    return torch.cat([lo * c - hi * s, lo * s + hi * c], -1)


def exact(case, seed):
    t = _tensors(case, seed)
    B, H, Hkv, L, S, D = (case[n] for n in ("B", "H", "Hkv", "L", "S", "D"))
    dt = DTYPES[case["dtype"]]
    if case["kind"] == "sdpa":
        k, v = t["k"], t["v"]
        if case["kv"] == "q8_0":
            k, v = (_q8_values(x, (B, Hkv, S, D)) for x in (k, v))
        mask = _mask(case, seed)
        return torch.stack([_attend64(t["q"][b].double(), k[b].double(), v[b].double(), _bias64(case, mask, b, L, S, DEV))[0]
                            for b in range(B)])
    if case["kind"] == "train":
        if case["dropout"]:
            return None  # the dropped positions are this package's own draw
        mask = _mask(case, seed)
        parts = []
        for b in range(B):
            q, k, v = (t[n][b].double().requires_grad_(True) for n in ("q", "k", "v"))
            out, _ = _attend64(q, k, v, _bias64(case, mask, b, L, S, DEV))
            parts.append([out.detach(), *torch.autograd.grad(out, (q, k, v), t["dout"][b].double())])
        return [torch.stack(x) for x in zip(*parts)]
    if case["kind"] == "cache":
        T = L + case["steps"]
        q = _rope64(t["q"], 0).to(dt).double()
        k, v = _rope64(t["k"], 0).to(dt), t["v"]  # rotated keys have the keys' dtype, then the cache's
        if case["kv"] == "q8_0":
            k, v = (_q8_values(_q8_blocks(x), x.shape) for x in (k, v))
        k, v = k.double(), v.double()
        bias = _bias64({"causal": True}, None, 0, T, T, DEV)
        out = torch.stack([_attend64(q[b], k[b], v[b], bias)[0] for b in range(B)])
        return [out[:, :, :L]] + [out[:, :, i:i + 1] for i in range(L, T)]
    # mha
    E = H * D
    x, wi, bi, wo, bo = (t[n].double().requires_grad_(True) for n in ("x", "w_in", "b_in", "w_out", "b_out"))
    mask = _mask(case, seed)
    rows, ws = [], []
    for b in range(B):
        q, k, v = (y.reshape(L, H, D).transpose(0, 1) for y in (x[b] @ wi.t() + bi).split(E, -1))
        bias = torch.zeros((1, S), dtype=torch.float64, device=DEV)
        if mask is not None:
            bias = bias.masked_fill(mask[b][None], -1e9)
        o, w = _attend64(q, k, v, bias)
        rows.append(o.transpose(0, 1).reshape(L, E) @ wo.t() + bo)
        ws.append(torch.stack(w).mean(0))
    out = torch.stack(rows)
    grads = torch.autograd.grad(out, (x, wi, bi, wo, bo), t["dout"].double())
    return [out.detach(), torch.stack(ws).detach(), *grads]
