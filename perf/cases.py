"""The calls that programs built on this library spend their time in, as cases a timing program can run.

A case is a dict of plain values with a "kind":

  matmul     one linear layer over GGUF blocks (litenn_amd.mul_mat_q) on m activation rows
  attention  the attention layer with its options (litenn_hip_flash_attn_ext), all heads of one call
  llama      a resident LLaMA decoder: a prompt, and `new` greedy tokens behind it
  layered    a resident layered decoder (Kulurax, Degedra): a prompt, then `steps` tokens fed one at a time, as
             a program that samples on the host does

listed() has the sizes the library's configurations and benchmark name, with fewer blocks of a model than it has
(all blocks are alike); draw() gives others of the same ranges.  Inputs come from a seed alone.  exact() computes
the same outputs in 64 bits with plain torch.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

import litenn_amd as ln
from litenn_amd import _lib, synth
from litenn_amd.formats import (DT_F16, DT_F32, DT_U8, F32, Q4_0, Q4_K, Q5_K, Q6_K, Q8_0, block_layout, row_bytes)
from litenn_amd.model import to_bfloat16

FORMATS = {"Q4_0": Q4_0, "Q8_0": Q8_0, "Q4_K": Q4_K, "Q5_K": Q5_K, "Q6_K": Q6_K}
VOCAB = 32000


def listed():
    return [
        # one token through one feed-forward matrix of an 8B-shape model: the library's headline call
        {"name": "matmul_1_row", "kind": "matmul", "fmt": "Q4_K", "n": 14336, "k": 4096, "m": 1, "precise": False},
        # a handful of sequences decoded together
        {"name": "matmul_3_rows", "kind": "matmul", "fmt": "Q8_0", "n": 4096, "k": 4096, "m": 3, "precise": False},
        # a short prompt through one matrix with Float32 operands
        {"name": "matmul_45_rows_f32", "kind": "matmul", "fmt": "Q6_K", "n": 4096, "k": 14336, "m": 45, "precise": True},
        # a long prompt through one matrix, Float16 operands
        {"name": "matmul_512_rows", "kind": "matmul", "fmt": "Q4_K", "n": 14336, "k": 4096, "m": 512, "precise": False},
        # the attention layer with mask, slopes, soft cap and sinks over a prompt
        {"name": "attention_options", "kind": "attention", "m": 200, "keys": 1000, "heads": 32, "kv_heads": 8, "dim": 128,
         "half": True, "softcap": 30.0, "alibi": True, "sinks": True},
        # a prompt as LLaMA.eval() runs it by default: Float32 operands
        {"name": "llama_prompt_f32", "kind": "llama", "shape": "8b", "width": 4096, "ff": 14336, "blocks": 2, "prompt": 300,
         "calls": 1, "new": 0, "precise": True},
        # a long prompt with Float16 operands, fed in two portions
        {"name": "llama_prompt_f16", "kind": "llama", "shape": "7b", "width": 4096, "ff": 11008, "blocks": 3, "prompt": 2048,
         "calls": 2, "new": 0, "precise": False},
        # greedy decoding on the device, defaults throughout
        {"name": "llama_generate", "kind": "llama", "shape": "8b", "width": 4096, "ff": 14336, "blocks": 3, "prompt": 20,
         "calls": 1, "new": 64, "precise": True},
        # layered decoders: a long and a middling prompt in the precision they are served with
        {"name": "kulurax_prompt", "kind": "layered", "design": "kulurax", "width": 4096, "layers": 2, "prompt": 2048,
         "steps": 0, "dtype": "bfloat16"},
        {"name": "degedra_prompt", "kind": "layered", "design": "degedra", "width": 2048, "layers": 3, "prompt": 777,
         "steps": 0, "dtype": "bfloat16"},
        # every operand in 32 bits
        {"name": "degedra_prompt_f32", "kind": "layered", "design": "degedra", "width": 2048, "layers": 2, "prompt": 500,
         "steps": 0, "dtype": "float32"},
        # one token at a time with the logits on the host
        {"name": "kulurax_steps", "kind": "layered", "design": "kulurax", "width": 4096, "layers": 2, "prompt": 3,
         "steps": 24, "dtype": "bfloat16"},
    ]


def _log_uniform(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["matmul", "matmul", "attention", "llama", "llama", "layered", "layered"])
    if kind == "matmul":
        fmt = rng.choice(sorted(FORMATS))
        k = 256 * _log_uniform(rng, 4, 56)
        if block_layout(FORMATS[fmt])[0] == 32 and rng.random() < 0.25:
            k += 32 * rng.randrange(1, 8)  # rows that are no whole number of 256-element chunks
        precise = rng.random() < 0.4
        return {"kind": kind, "fmt": fmt, "n": _log_uniform(rng, 500, 14336), "k": min(k, 14336),
                "m": _log_uniform(rng, 1, 64 if precise else 512), "precise": precise}
    if kind == "attention":
        keys = _log_uniform(rng, 60, 1100)
        return {"kind": kind, "m": min(keys, _log_uniform(rng, 4, 220)), "keys": keys, "heads": 32,
                "kv_heads": rng.choice([4, 8, 32]), "dim": rng.choice([64, 128, 128]), "half": rng.random() < 0.75,
                "softcap": rng.choice([0.0, 30.0]), "alibi": rng.random() < 0.5, "sinks": rng.random() < 0.5}
    if kind == "llama":
        width = rng.choice([1024, 2048, 4096])
        precise = rng.random() < 0.5
        return {"kind": kind, "shape": rng.choice(["7b", "8b", "q8"]), "width": width,
                "ff": 256 * rng.randint(int(width * 2.6) // 256, int(width * 3.5) // 256), "blocks": rng.randint(1, 2),
                "prompt": _log_uniform(rng, 6, 300 if precise else 2048), "calls": rng.choice([1, 1, 2]),
                "new": rng.choice([0, 0, rng.randint(8, 64)]) if precise else 0, "precise": precise}
    dtype = rng.choice(["bfloat16", "bfloat16", "float32"])
    steps = rng.choice([0, 0, rng.randint(4, 24)])
    width = rng.choice([1024, 2048, 4096] if dtype == "bfloat16" else [1024, 2048])
    return {"kind": kind, "design": rng.choice(["kulurax", "degedra"]), "width": width, "layers": 2,
            "prompt": rng.randint(1, 40) if steps else _log_uniform(rng, 16, 2048 if dtype == "bfloat16" else 500),
            "steps": steps, "dtype": dtype}


# ---- inputs ------------------------------------------------------------------------------------------

def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


# bytes of a block that hold Float16 scales
SCALES = {Q4_0: (0,), Q8_0: (0,), Q4_K: (0, 2), Q5_K: (0, 2), Q6_K: (208,)}


def _blocks(fmt, count, sigma, g):
    """uint8 [count, block bytes] on the GPU: uniform codes, Float16 scales of either sign with that spread."""
    size = block_layout(fmt)[1]
    raw = torch.randint(0, 1 << 31, ((count * size + 3) // 4 + 1,), generator=g, device="cuda", dtype=torch.int64)
    raw = (raw ^ (raw << 7)).to(torch.int32).view(torch.uint8)[:count * size].reshape(count, size).clone()
    if fmt == Q8_0:
        raw[:, 2:][raw[:, 2:] == 128] = 129  # a quantiser writes no -128
    for at in SCALES[fmt]:
        raw[:, at:at + 2] = (torch.randn(count, 1, generator=g, device="cuda") * sigma).half().view(torch.uint8)
    return raw


def _payload(fmt, n, k, g):
    """uint8 [n, row bytes] on the GPU; the dequantised matrix has entries of root mean square 1 / sqrt(k)."""
    return _blocks(fmt, n * k // block_layout(fmt)[0], 1.0 / (synth.CODE_RMS[fmt] * math.sqrt(k)), g).reshape(n, -1)


LLAMA_FORMATS = {"7b": {"default": Q4_0}, "q8": {"default": Q8_0},
                 "8b": {"default": Q4_K, "attn_v": Q6_K, "ffn_down": Q6_K, "output": Q6_K}}


def _llama_config(case):
    heads = case["width"] // 128
    return synth.LLaMAConfig(case["shape"], case["blocks"], case["width"], heads, heads if case["shape"] == "7b" else heads // 4,
                             case["ff"], VOCAB, case["prompt"] + case["new"] + 8,
                             rope_freq_base=5e5 if case["shape"] == "8b" else 1e4, formats=LLAMA_FORMATS[case["shape"]])


def _llama_tensors(case, seed):
    """(kind, layer, format, host payload, n, k) of every tensor; the matrices of one format are windows into one pool."""
    cfg, g = _llama_config(case), _generator(seed)
    rng = np.random.default_rng(int(seed))
    shapes = cfg.tensor_shapes()
    spare, pools = 4096, {}
    for kind, (n, k) in shapes.items():
        pools[cfg.fmt(kind)] = max(pools.get(cfg.fmt(kind), 0), n * k // block_layout(cfg.fmt(kind))[0])
    pools = {f: _blocks(f, count + spare, 1.0 / (synth.CODE_RMS[f] * math.sqrt(cfg.embedding_length)), g).cpu().numpy()
             for f, count in sorted(pools.items())}

    def matrix(kind):
        n, k = shapes[kind]
        f = cfg.fmt(kind)
        at, count = int(rng.integers(0, spare)), n * k // block_layout(f)[0]
        return f, pools[f][at:at + count].reshape(n, -1), n, k

    d = cfg.embedding_length

    def norm():
        return F32, rng.uniform(0.5, 1.5, d).astype(np.float32), 1, d

    for kind in ("token_embd", "output"):
        yield (kind, -1, *matrix(kind))
    yield ("output_norm", -1, *norm())
    for layer in range(cfg.block_count):
        for kind in synth.TENSOR_KINDS:
            yield (kind, layer, *matrix(kind))
        for kind in ("attn_norm", "ffn_norm"):
            yield (kind, layer, *norm())


def _layered_config(case):
    w = case["width"]
    common = {"width": w, "ff": w * 7 // 2 if w == 4096 else w * 11 // 4, "layers": case["layers"], "heads": w // 128, "vocab": VOCAB,
              "window": 1024}
    if case["design"] == "kulurax":
        return synth.kulurax_config(kv_rank=w // 8, q_rank=w * 3 // 8, gla_heads=w // 256, **common)
    return synth.degedra_config(kv_heads=w // 512, ssm_heads=w // 64, **common)


def _layered_weights(case, seed):
    """{name: bfloat16 bits or Float32 vector}; the large matrices are windows into one pool of N(0, 1 / width)."""
    cfg = _layered_config(case)
    rng, g = np.random.default_rng(int(seed)), _generator(seed)
    shapes = synth.TENSOR_SHAPES[cfg["architecture"]](cfg)
    large = 1 << 20
    pool = max(int(np.prod(s)) for n, s in shapes.items() if not n.startswith(("embed", "head")))
    pool = (torch.randn(pool + 65536, generator=g, device="cuda") * case["width"] ** -0.5).bfloat16().view(torch.int16)
    pool = pool.cpu().numpy().view(np.uint16)
    out = {}
    for name, s in shapes.items():
        leaf, count = name.rsplit(".", 1)[-1], int(np.prod(s))
        if name in ("embed", "head"):  # a tied table takes part in both ends: entries well below one
            scale = (0.2 if case["design"] == "kulurax" else 1.0) if name == "embed" else case["width"] ** -0.5
            t = (torch.randn(s, generator=g, device="cuda") * scale).bfloat16().view(torch.int16)
            out[name] = t.cpu().numpy().view(np.uint16)
        elif len(s) == 2 and count >= large:
            at = int(rng.integers(0, 65536))
            out[name] = pool[at:at + count].reshape(s)
        elif len(s) == 2:
            out[name] = to_bfloat16(rng.normal(0.0, s[1] ** -0.5, s))
        else:
            low, high = {"A_log": (-3.0, 1.0), "dt_bias": (-4.0, 1.0), "b": (-0.3, 0.3) if "conv" in name else (-1.0, 4.0),
                         "D": (-1.0, 1.0), "sink": (-1.0, 2.0)}.get(leaf, (0.5, 1.5))
            out[name] = rng.uniform(low, high, s).astype(np.float32)
    return out


def _tokens(count, seed):
    return np.random.default_rng([int(seed), 77]).integers(0, VOCAB, count).astype(np.int32)


def _attention_inputs(case, seed):
    g = _generator(seed)
    kv = torch.float16 if case["half"] else torch.float32

    def normal(*shape):
        return torch.randn(shape, generator=g, device="cuda")
    q = normal(case["m"], case["heads"] * case["dim"])
    k, v = (normal(case["keys"], case["kv_heads"] * case["dim"]).to(kv) for _ in range(2))
    mask = None
    if case["alibi"]:  # distances to the key, as an ALiBi caller passes them
        at = torch.arange(case["keys"], device="cuda", dtype=torch.float32)
        mask = -(at[None, :] - (case["keys"] - case["m"] + torch.arange(case["m"], device="cuda"))[:, None]).abs()
    sinks = normal(case["heads"]) if case["sinks"] else None
    return q, k, v, mask, sinks


class _Operand:
    """A torch tensor as the operand of the library's device functions."""

    def __init__(self, tensor, dtype):
        self.tensor, self.dtype, self.device = tensor, dtype, ln.HIP()
        self.ptr, self.size = tensor.data_ptr(), tensor.numel()


class _State:
    def __init__(self, **fields):
        self.__dict__.update(fields)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "matmul":
        g, fmt = _generator(seed), FORMATS[case["fmt"]]
        return _State(case=case, fmt=fmt, w=_Operand(_payload(fmt, case["n"], case["k"], g), DT_U8),
                      x=_Operand(torch.randn(case["m"], case["k"], generator=g, device="cuda"), DT_F32),
                      y=_Operand(torch.empty(case["m"], case["n"], device="cuda"), DT_F32))
    if kind == "attention":
        q, k, v, mask, sinks = _attention_inputs(case, seed)
        options = _lib.AttnExtOpts(case["dim"] ** -0.5, 8.0 if case["alibi"] else 0.0, case["softcap"],
                                   mask.data_ptr() if mask is not None else None,
                                   sinks.data_ptr() if sinks is not None else None, 1, 0, case["keys"] - case["m"])
        return _State(case=case, q=q, k=k, v=v, mask=mask, sinks=sinks, options=options, out=torch.empty_like(q))
    if kind == "llama":
        model = ln.LLaMA.from_config(_llama_config(case), kv_dtype=DT_F16)
        model.load(_llama_tensors(case, seed))
        return _State(case=case, model=model, tokens=_tokens(case["prompt"], seed))
    model = ln.create_model(_layered_config(case), _layered_weights(case, seed), dtype=case["dtype"],
                            context_length=case["prompt"] + case["steps"] + 8)
    return _State(case=case, model=model, tokens=_tokens(case["prompt"] + case["steps"], seed))


def _portions(tokens, calls):
    """The prompt in `calls` parts of about the same length."""
    return [p for p in np.array_split(tokens, calls) if p.size]


def run(s):
    case, kind = s.case, s.case["kind"]
    if kind == "matmul":
        ln.mul_mat_q(s.fmt, s.w, case["n"], case["k"], s.x, s.y, flags=ln.MATMUL_PRECISE if case["precise"] else 0,
                     synchronize=False)
        return s.y.tensor
    if kind == "attention":
        _lib.check(_lib.load().litenn_hip_flash_attn_ext(
            0, s.q.data_ptr(), s.k.data_ptr(), s.v.data_ptr(), DT_F16 if case["half"] else DT_F32, case["m"], case["keys"],
            case["heads"], case["kv_heads"], case["dim"], C.byref(s.options), s.out.data_ptr(), C.byref(_lib.Exec(None, 0))))
        return s.out
    s.model.reset()
    if kind == "llama":
        parts = _portions(s.tokens, case["calls"])
        for part in parts[:-1]:
            s.model.eval(part, all_logits=False, precise=case["precise"])
        if not case["new"]:
            return {"logits": s.model.eval(parts[-1], all_logits=False, precise=case["precise"])}
        tokens, _, _ = s.model.generate(parts[-1], case["new"], precise=case["precise"])
        return {"tokens": tokens, "logits": s.model.eval(tokens[-1:], all_logits=False, precise=case["precise"])}
    n = case["prompt"]
    rows = [s.model.eval(s.tokens[:n], want=[n - 1])]
    rows += [s.model.eval(s.tokens[n + i:n + i + 1]) for i in range(case["steps"])]
    return {"logits": np.concatenate(rows)}


# ---- what a pass cannot do without ------------------------------------------------------------------

def work(case):
    kind = case["kind"]
    if kind == "matmul":
        n, k, m = case["n"], case["k"], case["m"]
        return {"bytes": n * row_bytes(FORMATS[case["fmt"]], k) + 4 * m * (n + k), "flops": 2.0 * m * n * k}
    if kind == "attention":
        m, keys, heads, dim = case["m"], case["keys"], case["heads"], case["dim"]
        pairs = m * (keys - m) + m * (m + 1) / 2
        size = (2 if case["half"] else 4) * 2 * keys * case["kv_heads"] * dim + 8 * m * heads * dim
        return {"bytes": size + (4 * m * keys if case["alibi"] else 0), "flops": 4.0 * pairs * heads * dim}
    if kind == "llama":
        cfg = _llama_config(case)
        t, new, blocks = case["prompt"], case["new"], cfg.block_count
        weights = cfg.matmul_weight_bytes_per_token()
        macs = sum(n * k for kind, (n, k) in cfg.tensor_shapes().items() if kind not in ("token_embd", "output")) * blocks
        head = VOCAB * cfg.embedding_length
        rows = t + new
        cached = 4 * cfg.head_count_kv * cfg.head_dim * blocks
        reads = cached * (t + new * (t + new / 2))
        passes = case["calls"] + new
        return {"bytes": weights * passes + reads + cached * rows + 4 * VOCAB * (1 + new),
                "flops": 2.0 * macs * rows + 2.0 * head * passes + 2.0 * blocks * cfg.embedding_length * rows * (rows + 1)}
    cfg = _layered_config(case)
    weights, steps = synth.layered_decode_weight_bytes(cfg), case["steps"]
    head = 2.0 * VOCAB * cfg["width"]
    per_token = synth.layered_prefill_flops(cfg, 1) - head
    return {"bytes": weights * (1 + steps) + 4 * VOCAB * (1 + steps),
            "flops": synth.layered_prefill_flops(cfg, case["prompt"]) + (per_token + head) * steps}


def tolerance(case):
    """About four times what the library and exact() differ by."""
    kind = case["kind"]
    if kind == "matmul":
        # Float32 operands below four rows and on request (2e-7), otherwise operands rounded to Float16 once (3e-4)
        return {"rel": 2e-6} if case["precise"] or case["m"] < 4 else {"rel": 1.2e-3}
    if kind == "attention":
        return {"rel": 4e-6}
    if kind == "llama":
        # Float32 operands: what is left are cached Float16 values rounded to the other side (2e-4)
        return {"rel": 1e-3, "differ": 0.0} if case["precise"] else {"rel": 7e-3}
    return {"rel": 1.6e-2} if case["dtype"] == "bfloat16" else {"rel": 1.2e-5}


# ---- the same in 64 bits ------------------------------------------------------------------------------

def _half(raw):
    return raw.contiguous().view(torch.float16).double()


def _six_bit(s):
    low, mid, high = s[..., 0:4], s[..., 4:8], s[..., 8:12]
    scale = torch.cat([low & 63, (high & 15) | ((low >> 6) << 4)], -1)
    least = torch.cat([mid & 63, (high >> 4) | ((mid >> 6) << 4)], -1)
    return scale.double()[..., None], least.double()[..., None]


def _dequantised(fmt, raw, k):
    """float64 [rows, k] of uint8 [rows, row bytes]."""
    b = raw.reshape(raw.shape[0], -1, block_layout(fmt)[1])
    rows, nb = b.shape[:2]
    if fmt == Q4_0:
        q = b[..., 2:]
        out = (torch.cat([q & 15, q >> 4], -1).double() - 8) * _half(b[..., 0:2])
    elif fmt == Q8_0:
        out = b[..., 2:].contiguous().view(torch.int8).double() * _half(b[..., 0:2])
    elif fmt in (Q4_K, Q5_K):
        scale, least = _six_bit(b[..., 4:16])
        q = b[..., -128:].reshape(rows, nb, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 3).reshape(rows, nb, 8, 32).double()
        if fmt == Q5_K:
            bit = torch.arange(8, device=b.device, dtype=torch.uint8)[:, None]
            q = q + 16 * ((b[..., None, 16:48] >> bit) & 1).double()
        out = _half(b[..., 0:2])[..., None] * scale * q - _half(b[..., 2:4])[..., None] * least
    else:
        low = b[..., :128].reshape(rows, nb, 2, 1, 64)
        low = torch.cat([low & 15, low >> 4], 3).reshape(rows, nb, 2, 4, 32)
        shift = torch.tensor([0, 2, 4, 6], device=b.device, dtype=torch.uint8)[:, None]
        high = (b[..., 128:192].reshape(rows, nb, 2, 1, 32) >> shift) & 3
        q = (low.double() + 16 * high.double() - 32).reshape(rows, nb, 16, 16)
        out = _half(b[..., 208:210])[..., None] * b[..., 192:208].contiguous().view(torch.int8).double()[..., None] * q
    return out.reshape(rows, k)


def _rms(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _softmax_values(q, k, v, scale, first, window=None, sink=None):
    """q [T, H, D], k [L, G, D], v [L, G, E]; query i stands at position first + i of the keys."""
    t, heads, share = q.shape[0], q.shape[1], q.shape[1] // k.shape[1]
    i = first + torch.arange(t, device=q.device)[:, None]
    j = torch.arange(k.shape[0], device=q.device)[None, :]
    hidden = (j > i) if window is None else (j > i) | (i - j >= window)
    out = torch.empty(t, heads, v.shape[2], dtype=q.dtype, device=q.device)
    for h in range(heads):
        s = (q[:, h] @ k[:, h // share].T * scale).masked_fill(hidden, -math.inf)
        if sink is not None:
            s = torch.cat([s, sink[h].expand(t, 1)], 1)
        out[:, h] = torch.softmax(s, 1)[:, :k.shape[0]] @ v[:, h // share]
    return out


def _exact_attention(case, seed):
    q, k, v, mask, sinks = _attention_inputs(case, seed)
    m, keys, heads, kv, dim = case["m"], case["keys"], case["heads"], case["kv_heads"], case["dim"]
    q, k, v = q.double().view(m, heads, dim), k.double().view(keys, kv, dim), v.double().view(keys, kv, dim)
    hidden = torch.arange(keys, device="cuda")[None, :] > (keys - m + torch.arange(m, device="cuda"))[:, None]
    power = 1 << int(math.floor(math.log2(heads)))
    base, odd = 2.0 ** (-8.0 / power), 2.0 ** (-4.0 / power)
    out = torch.empty_like(q)
    for h in range(heads):
        s = q[:, h] @ k[:, h * kv // heads].T * dim ** -0.5
        if case["softcap"]:
            s = case["softcap"] * torch.tanh(s / case["softcap"])
        if mask is not None:
            s = s + mask.double() * (base ** (h + 1) if h < power else odd ** (2 * (h - power) + 1))
        s = s.masked_fill(hidden, -math.inf)
        if sinks is not None:
            s = torch.cat([s, sinks[h].double().expand(m, 1)], 1)
        out[:, h] = torch.softmax(s, 1)[:, :keys] @ v[:, h * kv // heads]
    return out.view(m, heads * dim)


class _ExactLlama:
    def __init__(self, case, seed):
        self.cfg = _llama_config(case)
        self.w = {}
        for kind, layer, fmt, payload, n, k in _llama_tensors(case, seed):
            t = torch.from_numpy(payload).cuda()
            self.w[kind, layer] = (fmt, t, k) if fmt != F32 else t.double()
        self.cache = [None] * self.cfg.block_count
        self.past = 0

    def linear(self, x, kind, layer):
        fmt, raw, k = self.w[kind, layer]
        parts = [x @ _dequantised(fmt, raw[i:i + 8192], k).T for i in range(0, raw.shape[0], 8192)]
        return torch.cat(parts, 1)

    def rotate(self, x):
        """x [T, H, D]: interleaved pairs, all features of a head."""
        n = self.cfg.head_dim
        at = self.past + torch.arange(x.shape[0], device=x.device, dtype=torch.float64)
        angle = at[:, None] * self.cfg.rope_freq_base ** (-2.0 * torch.arange(n // 2, device=x.device) / n)
        c, s = torch.cos(angle)[:, None], torch.sin(angle)[:, None]
        a, b = x[..., 0::2], x[..., 1::2]
        return torch.stack([a * c - b * s, a * s + b * c], -1).flatten(-2)

    def eval(self, tokens):
        cfg = self.cfg
        fmt, table, k = self.w["token_embd", -1]
        x = _dequantised(fmt, table[torch.from_numpy(np.asarray(tokens, np.int64)).cuda()], k)
        t, hd = x.shape[0], cfg.head_dim
        for i in range(cfg.block_count):
            h = _rms(x, self.w["attn_norm", i], cfg.rms_eps)
            q, keys, values = (self.linear(h, "attn_" + n, i).view(t, -1, hd) for n in "qkv")
            new = [a.half().double() for a in (self.rotate(keys), values)]  # the cache's type
            self.cache[i] = new if self.cache[i] is None else [torch.cat(p) for p in zip(self.cache[i], new)]
            o = _softmax_values(self.rotate(q), *self.cache[i], hd ** -0.5, self.past).flatten(1)
            x = x + self.linear(o, "attn_output", i)
            h = _rms(x, self.w["ffn_norm", i], cfg.rms_eps)
            h = torch.nn.functional.silu(self.linear(h, "ffn_gate", i)) * self.linear(h, "ffn_up", i)
            x = x + self.linear(h, "ffn_down", i)
        self.past += t
        return self.linear(_rms(x[-1:], self.w["output_norm", -1], cfg.rms_eps), "output", -1)[0]


def _exact_llama(case, seed):
    model = _ExactLlama(case, seed)
    for part in _portions(_tokens(case["prompt"], seed), case["calls"]):
        logits = model.eval(part)
    if not case["new"]:
        return {"logits": logits}
    tokens = []
    for _ in range(case["new"]):
        tokens.append(int(logits.argmax()))
        logits = model.eval(tokens[-1:])
    return {"tokens": torch.tensor(tokens, dtype=torch.int32), "logits": logits}


def _kulurax_mixer(kind, h, w, m, eps):
    t, heads, dim, vdim = h.shape[0], m["heads"], m["dim"], m["vdim"]
    if kind == "latent_attention":
        q = (_rms(h @ w("dq").T, w("dq.norm"), eps) @ w("uq").T).view(t, heads, dim)
        c = _rms(h @ w("dkv").T, w("dkv.norm"), eps)
        k, v = (c @ w("uk").T).view(t, heads, dim), (c @ w("uv").T).view(t, heads, vdim)
        o = _softmax_values(q, k, v, m["scale"], 0, m["mask"]["size"], w("sink")).flatten(1)
        return (o * torch.sigmoid(h @ w("g").T)) @ w("o").T
    q, k = (h @ w("q").T).view(t, heads, dim) * dim ** -0.5, (h @ w("k").T).view(t, heads, dim)
    v = (h @ w("v").T).view(t, heads, vdim)
    decay = torch.exp(torch.nn.functional.logsigmoid(h @ w("a1").T @ w("a2").T + w("a2.b")) / m["tau"]).view(t, heads, dim)
    state, o = torch.zeros(heads, dim, vdim, dtype=h.dtype, device=h.device), torch.empty_like(v)
    for i in range(t):
        state = decay[i][:, :, None] * state + k[i][:, :, None] * v[i][:, None, :]
        o[i] = (state * q[i][:, :, None]).sum(1)
    return (_rms(o, w("norm"), eps).flatten(1) * torch.nn.functional.silu(h @ w("g").T)) @ w("o").T


def _degedra_mixer(h, w, m, eps):
    a, r = m["left"], m["right"]
    t, heads, groups, dim = h.shape[0], a["heads"], a["kv_heads"], a["dim"]
    values = h @ w("left.k").T
    q = _rms(h @ w("left.q").T, w("left.q.norm"), eps).view(t, heads, dim)
    k = _rms(values, w("left.k.norm"), eps).view(t, groups, dim)
    half = a["rot"]["dims"] // 2
    at = torch.arange(t, device=h.device, dtype=torch.float64)[:, None]
    angle = at * float(a["rot"]["base"]) ** (-2.0 * torch.arange(half, device=h.device) / a["rot"]["dims"])
    c, s = torch.cos(angle)[:, None], torch.sin(angle)[:, None]

    def turn(x):
        u, v = x[..., :half], x[..., half:2 * half]
        return torch.cat([u * c - v * s, v * c + u * s, x[..., 2 * half:]], -1)
    o = _softmax_values(turn(q), turn(k), values.view(t, groups, dim), a["scale"], 0, a["mask"]["size"]).flatten(1)
    left = o @ w("left.o").T

    heads, vdim, n, groups = r["heads"], r["vdim"], r["state"], r["groups"]
    inner, p = heads * vdim, h @ w("right.in").T
    z, xbc, dt = p[:, :inner], p[:, inner:2 * inner + 2 * groups * n], p[:, 2 * inner + 2 * groups * n:]
    taps = w("right.conv")
    padded = torch.cat([xbc.new_zeros(r["conv"] - 1, xbc.shape[1]), xbc])
    xbc = torch.nn.functional.silu(sum(padded[i:i + t] * taps[:, i] for i in range(r["conv"])) + w("right.conv.b"))
    x = xbc[:, :inner].view(t, heads, vdim)
    spread = torch.arange(heads, device=h.device) // (heads // groups)
    b, c = (xbc[:, inner + i * groups * n:inner + (i + 1) * groups * n].view(t, groups, n)[:, spread] for i in range(2))
    dt = torch.nn.functional.softplus(dt + w("right.dt_bias"), threshold=700)
    decay = torch.exp(-torch.exp(w("right.A_log")) * dt)
    state, y = torch.zeros(heads, n, vdim, dtype=h.dtype, device=h.device), torch.empty_like(x)
    for i in range(t):
        state = decay[i][:, None, None] * state + (dt[i][:, None] * b[i])[:, :, None] * x[i][:, None, :]
        y[i] = (state * c[i][:, :, None]).sum(1)
    y = (y + w("right.D")[:, None] * x).reshape(t, inner) * torch.nn.functional.silu(z)
    y = _rms(y.view(t, r["norm_groups"], -1), 1.0, eps).reshape(t, inner) * w("right.norm")
    return m["left_scale"] * left + m["right_scale"] * (y @ w("right.o").T)


def _exact_layered(case, seed):
    cfg, weights = _layered_config(case), _layered_weights(case, seed)
    eps = cfg["norm"]["eps"]
    tokens = _tokens(case["prompt"] + case["steps"], seed)

    def wide(name):
        t = weights[name]
        if t.dtype == np.uint16:
            return torch.from_numpy(t.view(np.int16)).cuda().view(torch.bfloat16).double()
        return torch.from_numpy(t).cuda().double()

    silu = torch.nn.functional.silu
    x = wide("embed")[torch.from_numpy(tokens.astype(np.int64)).cuda()]
    t, width = x.shape
    if case["design"] == "kulurax":
        j = torch.arange(width, device=x.device)
        angle = torch.arange(t, device=x.device, dtype=torch.float64)[:, None] * 10000.0 ** (-2.0 * (j // 2) / width)
        x = x + torch.where(j % 2 == 0, torch.sin(angle), torch.cos(angle))
    for i, layer in enumerate(cfg["layers"]):
        def w(name, i=i):
            return wide("l%d.mix.%s" % (i, name))
        p = "l%d." % i
        if case["design"] == "kulurax":
            y = _kulurax_mixer(layer["type"], _rms(x, wide(p + "norm1"), eps), w, layer["mixer"], eps)
            x = x + _rms(y, wide(p + "norm1b"), eps)
            h, limit = _rms(x, wide(p + "norm2"), eps), layer["mlp"]["limit"]
            g = (h @ wide(p + "mlp.gate").T).clamp(max=limit)
            u = (h @ wide(p + "mlp.up").T).clamp(-limit, limit)
            x = x + _rms((g * torch.sigmoid(1.702 * g) * (u + 1.0)) @ wide(p + "mlp.down").T, wide(p + "norm2b"), eps)
        else:
            x = x + _rms(_degedra_mixer(x, w, layer["mixer"], eps), wide(p + "norm1"), eps)
            y = (silu(x @ wide(p + "mlp.gate").T) * (x @ wide(p + "mlp.up").T)) @ wide(p + "mlp.down").T
            x = x + _rms(y, wide(p + "norm2"), eps)
    x = _rms(x[case["prompt"] - 1:], wide("final.norm"), eps)
    if case["design"] == "kulurax":
        return {"logits": x @ wide("embed").T}
    cap = cfg["logit_softcap"]
    return {"logits": cap * torch.tanh(x @ wide("head").T / cap)}


def exact(case, seed):
    kind = case["kind"]
    if kind == "matmul":
        g, fmt = _generator(seed), FORMATS[case["fmt"]]
        w = _payload(fmt, case["n"], case["k"], g)
        x = torch.randn(case["m"], case["k"], generator=g, device="cuda").double()
        return x @ _dequantised(fmt, w, case["k"]).T
    return {"attention": _exact_attention, "llama": _exact_llama, "layered": _exact_layered}[kind](case, seed)
