"""The work that a user of the library has it do, as cases to be measured.

Every case goes through the public entry points (the C ABI of
include/aihost_hip.h through aihost_amd._native, and aihost_amd.llama), with
device tensors as the operands.  Kinds of case:

  matmul     aih_matmul_weights_q: one quantized weight times M activation
             rows, the call that every projection of a model comes down to
             (decode M = 1, small batches M = 2..8, prompts above)
  attention  aih_attention over a KV cache (one query: decode; more: prompt)
  layer      LlamaDecoder.layer: one whole decoder layer over `rows` rows at
             positions start.. of a filled KV cache
  dequant    aih_dequantize of a whole tensor
  prefill    LlamaDecoder.prefill of a prompt, all layers and the head
  decode     one captured decode step of the whole model at the end of a prompt

listed() names the ones that are always looked at, draw() gives others of the
same ranges, exact() computes a case in 64-bit floating point in plain torch.
"""
import math

import torch

from aihost_amd import _native as nat
from aihost_amd import compute, llama

TYPES = {"Q4_0": nat.Q4_0, "Q8_0": nat.Q8_0, "Q4_K": nat.Q4_K, "Q6_K": nat.Q6_K}
BLOCK = {"Q4_0": (32, 18), "Q8_0": (32, 34), "Q4_K": (256, 144), "Q6_K": (256, 210)}   # elements, bytes
HEAD_DIM = 128
SHAPE = llama.LLAMA_8B_SHAPE


# ---- the cases ---------------------------------------------------------------
def listed():
    return [
        # the smallest projection of the 8B shape, one token: latency
        {"name": "matvec_q8_0_4096x4096", "kind": "matmul", "type": "Q8_0", "n": 4096, "k": 4096, "m": 1},
        # the FFN up projection of a decode step (the headline matvec)
        {"name": "matvec_q4_k_14336x4096", "kind": "matmul", "type": "Q4_K", "n": 14336, "k": 4096, "m": 1},
        # the FFN down projection, four sequences decoded together
        {"name": "batch4_q6_k_4096x14336", "kind": "matmul", "type": "Q6_K", "n": 4096, "k": 14336, "m": 4},
        # eight sequences decoded together
        {"name": "batch8_q4_0_14336x4096", "kind": "matmul", "type": "Q4_0", "n": 14336, "k": 4096, "m": 8},
        # a short question to a chat model: an odd number of prompt rows
        {"name": "gemm_q6_k_4096x14336_m33", "kind": "matmul", "type": "Q6_K", "n": 4096, "k": 14336, "m": 33},
        # the ordinary prompt of the benchmark
        {"name": "gemm_q4_k_4096x4096_m512", "kind": "matmul", "type": "Q4_K", "n": 4096, "k": 4096, "m": 512},
        # a long prompt through the FFN up projection
        {"name": "gemm_q4_k_14336x4096_m2048", "kind": "matmul", "type": "Q4_K", "n": 14336, "k": 4096, "m": 2048},
        # causal attention of a long prompt
        {"name": "attention_prompt_2048", "kind": "attention", "n_q": 2048, "start": 0, "heads": 32, "kv": 8},
        # a vocabulary table dequantized for an fp32 operator
        {"name": "dequant_q6_k_32000x4096", "kind": "dequant", "type": "Q6_K", "n": 32000, "k": 4096},
        # one decode layer far into a conversation
        {"name": "layer_decode_at_4000", "kind": "layer", "rows": 1, "start": 4000},
        # the benchmark's prompt through the whole model
        {"name": "prefill_8b_512", "kind": "prefill", "tokens": 512},
        # the benchmark's decode step, with the logits of the next token
        {"name": "decode_8b_at_512", "kind": "decode", "tokens": 512},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["matmul", "layer", "attention", "dequant"], [6, 2, 2, 1])[0]
    if kind == "matmul":
        typ = rng.choice(sorted(TYPES))
        # K in whole super-blocks (or pairs of 32-element blocks), N any
        k = 256 * _log(rng, 4, 56) if typ.endswith("_K") else 64 * _log(rng, 16, 224)
        n = _log(rng, 1024, 32000)
        if rng.random() < 0.6:
            n = n // 128 * 128
        m = rng.choice([1, 1, 2, rng.randint(3, 8), rng.randint(3, 8), _log(rng, 9, 128), _log(rng, 9, 128),
                        _log(rng, 129, 2048), _log(rng, 129, 2048)])
        return {"kind": kind, "type": typ, "n": n, "k": k, "m": m}
    if kind == "layer":
        rows = rng.choice([1, 1, rng.randint(2, 8), _log(rng, 9, 128), _log(rng, 129, 2048)])
        start = rng.choice([0, _log(rng, 16, 6000)]) if rows > 8 else _log(rng, 16, 8000)
        return {"kind": kind, "rows": rows, "start": start}
    if kind == "attention":
        n_q = rng.choice([1, _log(rng, 9, 2048), _log(rng, 128, 2048)])
        start = _log(rng, 16, 16000) if n_q == 1 else rng.choice([0, 0, _log(rng, 16, 4000)])
        kv = rng.choice([4, 8, 8])
        return {"kind": kind, "n_q": n_q, "start": start, "heads": kv * rng.choice([1, 4, 4, 8]), "kv": kv}
    return {"kind": kind, "type": rng.choice(sorted(TYPES)), "n": _log(rng, 256, 32000), "k": 256 * _log(rng, 4, 56)}


# ---- packed weights, made on the GPU by the GGUF rules -------------------------
def _half_bytes(v):
    return v.to(torch.float16).contiguous().view(torch.uint8).reshape(*v.shape, 2)


def _pack(typ, w):
    """Rows of fp32 weights (n, k) -> packed blocks, uint8 (n, k / QK, bytes)."""
    n = w.shape[0]
    qk = BLOCK[typ][0]
    b = w.reshape(n, -1, qk)
    if typ == "Q8_0":
        d = b.abs().amax(-1) / 127
        q = torch.round(b / d.clamp_min(1e-30).unsqueeze(-1)).clamp(-127, 127).to(torch.int8)
        return torch.cat([_half_bytes(d), q.view(torch.uint8)], -1)
    if typ == "Q4_0":
        top = b.gather(-1, b.abs().argmax(-1, keepdim=True)).squeeze(-1)
        d = top / -8
        inv = torch.where(d == 0, torch.zeros_like(d), 1 / d).unsqueeze(-1)
        q = torch.floor(b * inv + 8.5).clamp(0, 15).to(torch.uint8)
        return torch.cat([_half_bytes(d), q[..., :16] | (q[..., 16:] << 4)], -1)
    if typ == "Q4_K":
        s = b.reshape(n, -1, 8, 32)
        lo = s.amin(-1).clamp_max(0)
        scale, low = (s.amax(-1) - lo) / 15, -lo
        d, dmin = scale.amax(-1) / 63, low.amax(-1) / 63
        sc = torch.round(scale / d.clamp_min(1e-30).unsqueeze(-1)).clamp(0, 63)
        mn = torch.round(low / dmin.clamp_min(1e-30).unsqueeze(-1)).clamp(0, 63)
        step = (d.half().float().unsqueeze(-1) * sc).clamp_min(1e-30).unsqueeze(-1)
        q = torch.round((s + (dmin.half().float().unsqueeze(-1) * mn).unsqueeze(-1)) / step).clamp(0, 15).to(torch.uint8)
        sc, mn = sc.to(torch.uint8), mn.to(torch.uint8)
        head = torch.cat([sc[..., :4] | ((sc[..., 4:] >> 4) << 6), mn[..., :4] | ((mn[..., 4:] >> 4) << 6),
                          (sc[..., 4:] & 15) | ((mn[..., 4:] & 15) << 4)], -1)
        qs = q[..., 0::2, :] | (q[..., 1::2, :] << 4)
        return torch.cat([_half_bytes(d), _half_bytes(dmin), head, qs.reshape(n, -1, 128)], -1)
    s = b.reshape(n, -1, 16, 16)
    top = s.gather(-1, s.abs().argmax(-1, keepdim=True)).squeeze(-1)
    scale = top / -32
    d = scale.abs().amax(-1) / 127
    sc = torch.round(scale / d.clamp_min(1e-30).unsqueeze(-1)).clamp(-127, 127)
    step = (d.half().float().unsqueeze(-1) * sc).unsqueeze(-1)
    inv = torch.where(step == 0, torch.zeros_like(step), 1 / step)
    q = (torch.round(s * inv).clamp(-32, 31) + 32).to(torch.uint8).reshape(n, -1, 2, 4, 32)
    ql = (q[..., 0:2, :] & 15) | ((q[..., 2:4, :] & 15) << 4)
    qh = (q[..., 0, :] >> 4) | ((q[..., 1, :] >> 4) << 2) | ((q[..., 2, :] >> 4) << 4) | ((q[..., 3, :] >> 4) << 6)
    return torch.cat([ql.reshape(n, -1, 128), qh.reshape(n, -1, 64), sc.to(torch.int8).view(torch.uint8),
                      _half_bytes(d)], -1)


def _unpack(typ, p):
    """Packed blocks -> float64 weights (n, k), the GGUF formulas in 64 bits."""
    n = p.shape[0]

    def half(x):
        return x.contiguous().view(torch.float16).double()

    if typ == "Q8_0":
        return (half(p[..., :2]) * p[..., 2:].contiguous().view(torch.int8).double()).reshape(n, -1)
    if typ == "Q4_0":
        q = torch.cat([p[..., 2:] & 15, p[..., 2:] >> 4], -1).double() - 8
        return (half(p[..., :2]) * q).reshape(n, -1)
    if typ == "Q4_K":
        a, b, c = p[..., 4:8], p[..., 8:12], p[..., 12:16]
        sc = torch.cat([a & 63, (c & 15) | ((a >> 6) << 4)], -1).double()
        mn = torch.cat([b & 63, (c >> 4) | ((b >> 6) << 4)], -1).double()
        qs = p[..., 16:].reshape(n, -1, 4, 32)
        q = torch.stack([qs & 15, qs >> 4], -2).reshape(n, -1, 8, 32).double()
        return ((half(p[..., 0:2]) * sc).unsqueeze(-1) * q - (half(p[..., 2:4]) * mn).unsqueeze(-1)).reshape(n, -1)
    ql, qh = p[..., :128].reshape(n, -1, 2, 2, 32), p[..., 128:192].reshape(n, -1, 2, 32)
    hi = torch.stack([(qh >> (2 * i)) & 3 for i in range(4)], -2)
    q = (torch.cat([ql & 15, ql >> 4], -2) | (hi << 4)).double().reshape(n, -1, 16, 16) - 32
    sc = p[..., 192:208].contiguous().view(torch.int8).double()
    return ((half(p[..., 208:210]) * sc).unsqueeze(-1) * q).reshape(n, -1)


class _Make:
    """Inputs from a seed: a torch generator on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed) * 7919 + 17)

    def normal(self, *shape):
        return torch.randn(*shape, generator=self.g, device="cuda", dtype=torch.float32)

    def ids(self, count, top):
        return torch.randint(0, top, (count,), generator=self.g, device="cuda", dtype=torch.int32)

    def packed(self, typ, n, k):
        """An n x k weight of N(0, 0.02) values, quantized."""
        parts = []
        for at in range(0, n, 8192):
            parts.append(_pack(typ, 0.02 * self.normal(min(8192, n - at), k)))
        return torch.cat(parts, 0)


# ---- one device and its stream for the whole program ---------------------------
_device = None


def device():
    global _device
    if _device is None:
        torch.cuda.init()
        _device = compute.HipComputeDevice(0)
    return _device


class _Owner:
    """Library objects, given back when nothing refers to them any more."""

    def __init__(self, *objects):
        self.objects = objects

    def __del__(self):
        if nat is not None and nat.lib is not None:   # not at the interpreter's end
            for o in self.objects:
                o.dispose()


class _Memory:
    """A library buffer seen as a tensor (no copy); it keeps its owner."""

    def __init__(self, owner, ptr, shape):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f4", "data": (int(ptr), False),
                                         "version": 2}


def _view(owner, ptr, *shape):
    return torch.as_tensor(_Memory(owner, ptr, shape), device="cuda")


class _State:
    """What a program holds."""

    def __init__(self, **kw):
        self.__dict__.update(kw)


# ---- inputs ----------------------------------------------------------------------
def _layer_weights(make, cfg, pre):
    """The weights of one layer of the 8B shape, packed on the GPU:
    {name: (type, tensor, rows, cols)}."""
    out = {}
    for suf, qt, r, c in llama.layer_tensors(cfg):
        if qt == nat.F32:
            out[pre + suf] = ("F32", 1.0 + 0.02 * make.normal(r * c), r, c)
        else:
            out[pre + suf] = ("Q4_K", make.packed("Q4_K", r, c), r, c)
    return out


def _model_weights(make, cfg, sets=2):
    """Weights of the whole model; layer l holds set l % sets."""
    made = [_layer_weights(make, cfg, "") for _ in range(sets)]
    out = {"token_embd": ("Q4_K", make.packed("Q4_K", cfg.vocab, cfg.dim), cfg.vocab, cfg.dim)}
    for l in range(cfg.n_layers):
        for suf, t in made[l % sets].items():
            out["blk.%d.%s" % (l, suf)] = t
    out["output_norm"] = ("F32", 1.0 + 0.02 * make.normal(cfg.dim), 1, cfg.dim)
    out["output"] = ("Q6_K", make.packed("Q6_K", cfg.vocab, cfg.dim), cfg.vocab, cfg.dim)
    return out


def _to_host(weights):
    """The form that DeviceWeights loads: ggml ids and host arrays."""
    seen, out = {}, {}
    for name, (typ, t, r, c) in weights.items():
        if id(t) not in seen:
            seen[id(t)] = t.cpu().numpy().reshape(-1)
        out[name] = (nat.F32 if typ == "F32" else TYPES[typ], seen[id(t)], r, c)
    return out


def _inputs(case, seed):
    """Every input of a case as tensors; prepare() and exact() both start here."""
    make = _Make(seed)
    kind = case["kind"]
    if kind == "matmul":
        return {"w": make.packed(case["type"], case["n"], case["k"]), "x": make.normal(case["m"], case["k"])}
    if kind == "dequant":
        return {"w": make.packed(case["type"], case["n"], case["k"])}
    if kind == "attention":
        n, end = case["n_q"], case["start"] + case["n_q"]
        return {"q": make.normal(n, case["heads"] * HEAD_DIM), "k": make.normal(end, case["kv"] * HEAD_DIM),
                "v": make.normal(end, case["kv"] * HEAD_DIM)}
    if kind == "layer":
        return {"x": make.normal(case["rows"], SHAPE.dim), "w": _layer_weights(make, SHAPE, "blk.0."),
                "k": make.normal(case["start"], SHAPE.kv_dim), "v": make.normal(case["start"], SHAPE.kv_dim)}
    ids = make.ids(case["tokens"] + 1, SHAPE.vocab)
    return {"ids": ids, "w": _model_weights(make, SHAPE)}


def _one_layer(cfg):
    return llama.LlamaConfig(n_layers=1, dim=cfg.dim, n_heads=cfg.n_heads, n_kv_heads=cfg.n_kv_heads,
                             head_dim=cfg.head_dim, ffn=cfg.ffn, vocab=cfg.vocab, eps=cfg.eps, theta=cfg.theta)


def prepare(case, seed):
    dev, L = device(), nat.lib()
    kind, data = case["kind"], _inputs(case, seed)
    s = _State(kind=kind, h=dev.handle, L=L)
    if kind == "matmul":
        s.w, s.x = data["w"], data["x"]
        s.y = torch.zeros(case["m"], case["n"], device="cuda")
        s.args = (s.h, TYPES[case["type"]], s.w.data_ptr(), case["n"], case["k"], s.x.data_ptr(), case["m"],
                  s.y.data_ptr())
    elif kind == "dequant":
        s.w = data["w"]
        s.y = torch.zeros(case["n"], case["k"], device="cuda")
        s.args = (s.h, TYPES[case["type"]], s.w.data_ptr(), s.y.data_ptr(), s.y.numel(), nat.F16_IEEE)
    elif kind == "attention":
        s.q, s.k, s.v = data["q"], data["k"], data["v"]
        rows = s.k.shape[0]
        s.y = torch.zeros_like(s.q)
        floats = int(L.aih_attention_scratch_floats(case["heads"], rows))
        s.scratch = torch.zeros(max(4, floats), device="cuda")
        s.args = (s.h, s.q.data_ptr(), s.k.data_ptr(), s.v.data_ptr(), s.y.data_ptr(), case["n_q"], case["heads"],
                  case["kv"], HEAD_DIM, case["start"], None, rows, 1.0 / math.sqrt(HEAD_DIM), s.scratch.data_ptr(),
                  floats)
    elif kind == "layer":
        rows, start, end = case["rows"], case["start"], case["start"] + case["rows"]
        w = llama.DeviceWeights(dev, _to_host(data["w"]))
        s.d = llama.LlamaDecoder(dev, _one_layer(SHAPE), w, end, rows)
        s.owner = _Owner(s.d, w)
        s.x, s.rows, s.start = data["x"], rows, start
        torch.cuda.synchronize()
        for to, src in ((s.d.kc[0], data["k"]), (s.d.vc[0], data["v"])):
            if start:
                nat.check(L.aih_memcpy_d2d(s.h, to, src.data_ptr(), src.numel() * 4), "cache rows")
        at = start * SHAPE.kv_dim * 4
        s.out = (_view(s.owner, s.d.x, rows, SHAPE.dim), _view(s.owner, s.d.kc[0] + at, rows, SHAPE.kv_dim),
                 _view(s.owner, s.d.vc[0] + at, rows, SHAPE.kv_dim))
    else:
        w = llama.DeviceWeights(dev, _to_host(data["w"]))
        s.n = case["tokens"]
        s.d = llama.LlamaDecoder(dev, SHAPE, w, s.n + 64, s.n)
        s.owner = _Owner(s.d, w)
        s.ids = data["ids"].cpu().numpy()
        s.out = _view(s.owner, s.d.logits, SHAPE.vocab)
        if kind == "decode":
            # the prompt's cache and the captured step; the token that follows
            # the prompt is given (as when a known text is scored), so that a
            # pass does not depend on a tie between two logits
            s.d.prefill(s.ids[:s.n])
            s.d.capture()
            s.token = data["ids"][s.n:].clone()
            s.pos = torch.full((1,), s.n, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    return s


def run(s):
    L = s.L
    if s.kind == "matmul":
        nat.check(L.aih_matmul_weights_q(*s.args), "aih_matmul_weights_q")
        return s.y
    if s.kind == "dequant":
        nat.check(L.aih_dequantize(*s.args), "aih_dequantize")
        return s.y
    if s.kind == "attention":
        nat.check(L.aih_attention(*s.args), "aih_attention")
        return s.y
    if s.kind == "layer":
        # the layer adds into its activation rows: they start from the input
        nat.check(L.aih_memcpy_d2d(s.h, s.d.x, s.x.data_ptr(), s.x.numel() * 4), "x")
        s.d.layer(0, s.rows, s.start, None)
        return s.out
    if s.kind == "prefill":
        s.d.prefill(s.ids[:s.n], read=False)
        return s.out
    nat.check(L.aih_memcpy_d2d(s.h, s.d.token, s.token.data_ptr(), 4), "token")
    nat.check(L.aih_memcpy_d2d(s.h, s.d.pos, s.pos.data_ptr(), 4), "position")
    nat.check(L.aih_graph_launch(s.h, s.d.capture()), "aih_graph_launch")
    return s.out


# ---- what a pass cannot do without -------------------------------------------------
def _layer_work(cfg, rows, start):
    weights = flops = 0
    for _, qt, r, c in llama.layer_tensors(cfg):
        weights += r * c * 4 if qt == nat.F32 else r * c // 256 * 144
        flops += 0 if qt == nat.F32 else 2 * rows * r * c
    keys = rows * start + rows * (rows + 1) // 2
    flops += 4 * keys * cfg.n_heads * cfg.head_dim
    cache = 2 * (start + rows) * cfg.kv_dim * 4
    return weights, cache, flops


def work(case):
    kind = case["kind"]
    if kind in ("matmul", "dequant"):
        n, k = case["n"], case["k"]
        qk, size = BLOCK[case["type"]]
        w = n * k // qk * size
        if kind == "dequant":
            return {"bytes": w + 4 * n * k, "flops": 2 * n * k}
        m = case["m"]
        return {"bytes": w + 4 * m * k + 4 * m * n, "flops": 2 * m * n * k}
    if kind == "attention":
        n, st = case["n_q"], case["start"]
        keys = n * st + n * (n + 1) // 2
        return {"bytes": 4 * HEAD_DIM * (2 * n * case["heads"] + 2 * (st + n) * case["kv"]),
                "flops": 4 * keys * case["heads"] * HEAD_DIM}
    if kind == "layer":
        w, cache, flops = _layer_work(SHAPE, case["rows"], case["start"])
        return {"bytes": w + cache + 8 * case["rows"] * SHAPE.dim, "flops": flops}
    rows, start = (case["tokens"], 0) if kind == "prefill" else (1, case["tokens"])
    w, cache, flops = _layer_work(SHAPE, rows, start)
    head = SHAPE.vocab * SHAPE.dim
    return {"bytes": SHAPE.n_layers * (w + cache) + head // 256 * 210 + rows * SHAPE.dim // 256 * 144 + 4 * SHAPE.vocab,
            "flops": SHAPE.n_layers * flops + 2 * head}


def tolerance(case):
    """Four times and more what the path shows against exact(): fp32
    arithmetic up to 8 activation rows (and in attention), fp16 operands with
    fp32 sums in the products of more rows, and in the whole model these
    through 32 layers."""
    kind = case["kind"]
    if kind == "dequant":
        return "exact"
    if kind == "attention":
        return {"rel": 1e-5, "max": 1e-3}
    if kind == "matmul":
        return {"rel": 1e-5, "max": 1e-3} if case["m"] <= 8 else {"rel": 1.5e-3, "max": 2e-2}
    if kind == "layer":
        # up to 8 rows the keys differ most: 2e-5 for an angle of one fp32
        # rounding more at a position of some thousands
        return {"rel": 8e-5, "max": 4e-3} if case["rows"] <= 8 else {"rel": 2e-3, "max": 4e-2}
    return {"rel": 2e-2, "max": 2e-1}


# ---- the same in 64 bits, without the library ---------------------------------------
def _attend(q, k, v, start, heads, kv):
    """Causal grouped-query attention: q (n, heads * d), cache rows k, v."""
    n, end = q.shape[0], k.shape[0]
    out = torch.empty_like(q)
    mask = torch.arange(end, device=q.device)[None, :] > (start + torch.arange(n, device=q.device))[:, None]
    for h in range(heads):
        g = h // (heads // kv)
        c, at = slice(g * HEAD_DIM, (g + 1) * HEAD_DIM), slice(h * HEAD_DIM, (h + 1) * HEAD_DIM)
        t = (q[:, at] @ k[:, c].T.contiguous() / math.sqrt(HEAD_DIM)).masked_fill(mask, -math.inf)
        out[:, at] = torch.softmax(t, -1) @ v[:, c].contiguous()
    return out


def _rope(x, start, theta):
    """Interleaved pairs; the angle is the fp32 product of position and frequency."""
    n, d = x.shape[0], HEAD_DIM
    freq = (1.0 / theta ** (torch.arange(0, d, 2, device=x.device, dtype=torch.float64) / d)).float()
    ang = (torch.arange(start, start + n, device=x.device).float()[:, None] * freq[None, :]).double()
    p = x.reshape(n, -1, d // 2, 2)
    c, s = torch.cos(ang)[:, None, :], torch.sin(ang)[:, None, :]
    return torch.stack([p[..., 0] * c - p[..., 1] * s, p[..., 0] * s + p[..., 1] * c], -1).reshape(x.shape)


def _norm(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


class _Dense:
    """Weights of a layer in 64 bits, unpacked once each."""

    def __init__(self, weights):
        self.w, self.seen = weights, {}

    def __getitem__(self, name):
        typ, t = self.w[name][:2]
        if id(t) not in self.seen:
            self.seen[id(t)] = t.double() if typ == "F32" else _unpack(typ, t)
        return self.seen[id(t)]


def _layer64(x, w, pre, k_old, v_old, start):
    c = SHAPE
    n = _norm(x, w[pre + "attn_norm"], c.eps)
    q = _rope(n @ w[pre + "attn_q"].T, start, c.theta)
    k = _rope(n @ w[pre + "attn_k"].T, start, c.theta)
    v = n @ w[pre + "attn_v"].T
    o = _attend(q, torch.cat([k_old, k]), torch.cat([v_old, v]), start, c.n_heads, c.n_kv_heads)
    x = x + o @ w[pre + "attn_output"].T
    n = _norm(x, w[pre + "ffn_norm"], c.eps)
    g = n @ w[pre + "ffn_gate"].T
    return x + (g * torch.sigmoid(g) * (n @ w[pre + "ffn_up"].T)) @ w[pre + "ffn_down"].T, k, v


def exact(case, seed):
    kind, data = case["kind"], _inputs(case, seed)
    if kind == "matmul":
        return data["x"].double() @ _unpack(case["type"], data["w"]).T
    if kind == "dequant":
        return _unpack(case["type"], data["w"])
    if kind == "attention":
        return _attend(data["q"].double(), data["k"].double(), data["v"].double(), case["start"], case["heads"],
                       case["kv"])
    w = _Dense(data["w"])
    if kind == "layer":
        return _layer64(data["x"].double(), w, "blk.0.", data["k"].double(), data["v"].double(), case["start"])
    ids = data["ids"].long()
    if kind == "prefill":
        ids = ids[:case["tokens"]]
    x = _unpack("Q4_K", data["w"]["token_embd"][1][ids])
    none = torch.zeros(0, SHAPE.kv_dim, device="cuda", dtype=torch.float64)
    for l in range(SHAPE.n_layers):
        x = _layer64(x, w, "blk.%d." % l, none, none, 0)[0]
    return _norm(x[-1:], w["output_norm"], SHAPE.eps)[0] @ w["output"].T
