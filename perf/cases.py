"""The performance cases of the framework: what a program that serves Qwen3-shaped models with it calls, over the ranges
it calls it in.

Three kinds of case:
  q8 / kq   one quantized matmul on device buffers (gw_q8_matmul, gw_kq_matmul): M activation rows by an N x K matrix
  step      one pass of a model (rq_decode, rq_forward_batch, rq_prefill): each sequence holds `len` positions and takes
            `new` tokens; the logits of each sequence's last row come back
The models have the widths of the repository's own workloads (8B Q8_0, 4B Q4_K_M, 0.6B Q8_0), the two wide ones with 4
layers and a vocabulary of 16,384 so that a pass is made of decoder layers and a state is made in seconds. Their weights
are seeded by the shape alone and loaded once per process, as a program keeps its model; tokens and caches follow the
case's seed. Every result of the framework is fixed bit for bit by its definition (a row's logits do not depend on its
batch, kernel or split), so the tolerance of every case is "exact".
"""
import math
import os
import tempfile

import numpy as np
import torch

import gwenedeg_amd as gw
from gwenedeg_amd import synth

WIDTHS = {  # model: (synthetic shape, layers, vocabulary, file bytes per weight in a layer)
    "8b": ("qwen3_8b", 4, 16384, 34 / 32),
    "4b": ("qwen3_4b_q4km", 4, 16384, 0.633),  # (Q4_K 144 / 256, Q6_K 210 / 256 on v and down)
    "0.6b": ("qwen3_0_6b", 28, 151936, 34 / 32),
}
KV = {"f16": gw.RQ_KV_F16, "bf16": gw.RQ_KV_BF16, "q8": gw.RQ_KV_Q8}
KV_BYTES = {"f16": 2.0, "bf16": 2.0, "q8": 17 / 16}
CTX = 36864  # the longest context a case uses, with room to grow
Q4_K, Q5_K = 12, 13
KQ_BYTES = {Q4_K: 144, Q5_K: 176}
DEV = "cuda"


def _step(name, model, lens, new, kv="f16", fill="synthetic"):
    """A pass over sequences of lens positions taking new tokens each (lists as comma-joined texts)."""
    return {"name": name, "kind": "step", "model": model, "lens": ",".join(map(str, lens)), "new": ",".join(map(str, new)),
            "kv": kv, "fill": fill}


def listed():
    mixed = [256 + (7936 * i * 7) // (48 * 7) + 13 * (i % 5) for i in range(48)]
    return [
        # the isolated Q8_0 operator at the repository's own size: one row (decode), a full prompt chunk
        {"name": "q8_12288x4096_m1", "kind": "q8", "n": 12288, "k": 4096, "m": 1},
        {"name": "q8_12288x4096_m512", "kind": "q8", "n": 12288, "k": 4096, "m": 512},
        # the K-quant operator over a prompt chunk (a 4B FFN matrix)
        {"name": "q4k_9728x2560_m512", "kind": "kq", "type": Q4_K, "n": 9728, "k": 2560, "m": 512},
        # chat decode: one sequence, a short context; the smallest model (launches and latency), the 8B and the 4B widths
        _step("decode_0.6b", "0.6b", [200], [1], fill="prompt"),
        _step("decode_8b", "8b", [577], [1], fill="prompt"),
        _step("decode_4b_q4km", "4b", [701], [1], fill="prompt"),
        # one long conversation: decode behind 32k cached positions
        _step("decode_8b_32k", "8b", [32701], [1]),
        # a serving batch: 32 sequences with 2,048 cached positions, a token each
        _step("batch32_4b_2k", "4b", [2048] * 32, [1] * 32),
        # long-context serving: 8 sequences with 32,768 cached positions
        _step("batch8_8b_32k", "8b", [32768] * 8, [1] * 8),
        # continuous batching: 48 decode rows at lengths 256 .. 8,192 beside prompt chunks of two new requests (one
        # behind a shared prefix of 1,024 positions)
        _step("mixed_8b", "8b", mixed + [0, 1024], [1] * 48 + [232, 232]),
        # prompts: a long one of odd length from nothing, a chunk behind 8k positions
        _step("prefill_4b_1537", "4b", [0], [1537], fill="prompt"),
        _step("prefill_8b_at_8k", "8b", [8192], [512]),
    ]


def _logu(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["q8", "kq", "decode", "decode", "batch", "batch", "prefill", "prefill", "mixed"])
    if kind == "q8":
        return {"kind": "q8", "n": 16 * _logu(rng, 64, 1536), "k": 32 * _logu(rng, 32, 384), "m": _logu(rng, 1, 512)}
    if kind == "kq":
        return {"kind": "kq", "type": rng.choice([Q4_K, Q4_K, Q5_K]), "n": 16 * _logu(rng, 64, 1024),
                "k": 256 * _logu(rng, 4, 40), "m": _logu(rng, 1, 512)}
    kv = rng.choice(["f16", "f16", "f16", "bf16", "q8"])
    model = rng.choice(["8b", "8b", "4b", "4b", "0.6b"])
    if kind == "decode":
        c = _step("", model, [_logu(rng, 16, 32000 if model != "0.6b" else 4000)], [1], kv)
    elif kind == "batch":
        n = _logu(rng, 2, 48 if model != "0.6b" else 8)
        top = min(32000, 200000 // n) if model != "0.6b" else min(4000, 60000 // n)
        c = _step("", model, [_logu(rng, 64, top) for _ in range(n)], [1] * n, kv)
    elif kind == "prefill":
        c = _step("", model, [rng.choice([0, 0, _logu(rng, 16, 6000)])], [_logu(rng, 2, 512)], kv)
    else:
        n, model = rng.randint(4, 40), rng.choice(["8b", "4b"])
        c = _step("", model, [_logu(rng, 64, 6000) for _ in range(n)] + [0], [1] * n + [_logu(rng, 16, 400)], kv)
    del c["name"]
    return c


def _lists(case):
    return [int(v) for v in case["lens"].split(",")], [int(v) for v in case["new"].split(",")]


def _shape(model):
    name, layers, vocab, wb = WIDTHS[model]
    d = dict(synth.SHAPES[name], n_layers=layers, vocab=vocab)
    return d, wb


_models = {}


def _write(model, d):
    return synth.write_gguf(os.path.join(d, model + ".gguf"), _shape(model)[0], seed=17)


def _model(model):
    if model not in _models:
        with tempfile.TemporaryDirectory() as d:
            _models[model] = gw.Model(_write(model, d), ctx_len=CTX)
    return _models[model]


def _tokens(seed, vocab, n):
    return np.random.default_rng([seed, 3]).integers(0, vocab, n).astype(np.int32)


def _op_inputs(case, seed):
    """Activation codes and scales as the quantizer makes them of N(0, 1) rows, weights as random codes and scales."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    n, k, m = case["n"], case["k"], case["m"]
    x = torch.randn(m, k // 32, 32, generator=g, device=DEV)
    top = x.abs().amax(-1, keepdim=True)
    s = {"xq": torch.clamp(torch.round(x * (127 / top)), -127, 127).to(torch.int8).reshape(m, k).contiguous(),
         "xs": (top[..., 0] / 127).contiguous()}
    if case["kind"] == "q8":
        s["codes"] = torch.randint(-127, 128, (n, k), generator=g, device=DEV, dtype=torch.int8)
        s["scales"] = (torch.randn(n, k // 32, generator=g, device=DEV).abs() * 1e-3).half()
    else:
        size = KQ_BYTES[case["type"]]
        b = torch.randint(0, 256, (n * (k // 256), size), generator=g, device=DEV, dtype=torch.uint8)
        d = (torch.rand(b.shape[0], 2, generator=g, device=DEV) * 1e-4 + 1e-5).half()
        b[:, :4] = d.view(torch.uint8)
        s["blocks"] = b.contiguous()
    return s


def prepare(case, seed):
    if case["kind"] != "step":
        s = _op_inputs(case, seed)
        s["out"] = torch.empty(case["m"], case["n"], device=DEV)
        return dict(s, case=case, stream=torch.cuda.current_stream().cuda_stream)
    lens, new = _lists(case)
    model = _model(case["model"])
    rows = sum(new)
    tok = _tokens(seed, model.vocab, sum(lens) + rows)
    ctx = model.ctx(max_batch=min(512, max(rows, 2)), max_ctx=max(a + b for a, b in zip(lens, new)))
    fill = model.ctx(max_batch=512, max_ctx=max(lens)) if case["fill"] == "prompt" and max(lens) else None
    seqs, parts, o = [], [], 0
    for i, (have, n) in enumerate(zip(lens, new)):
        s = model.seq(have + n, KV[case["kv"]])
        if have and fill:
            fill.prefill(s, tok[o:o + have], gw.RQ_LOGITS_NONE)
        elif have:
            s.fill_synthetic(have, _fill_seed(seed, i))
        seqs.append(s)
        parts.append(tok[o + have:o + have + n])
        o += have + n
    return {"case": case, "ctx": ctx, "seqs": seqs, "tokens": parts, "lens": lens}


def _fill_seed(seed, i):
    return 1 + 1009 * (seed % 1000003) + 7 * i


def run(state):
    case = state["case"]
    if case["kind"] == "q8":
        r = gw.lib.gw_q8_matmul(state["out"].data_ptr(), state["codes"].data_ptr(), state["scales"].data_ptr(), case["n"], case["k"],
                                state["xq"].data_ptr(), state["xs"].data_ptr(), case["m"], state["stream"])
    elif case["kind"] == "kq":
        r = gw.lib.gw_kq_matmul(state["out"].data_ptr(), case["type"], state["blocks"].data_ptr(), case["n"], case["k"],
                                state["xq"].data_ptr(), state["xs"].data_ptr(), case["m"], state["stream"])
    else:
        ctx, seqs, tokens = state["ctx"], state["seqs"], state["tokens"]
        for s, n in zip(seqs, state["lens"]):
            s.truncate(n)
        if len(seqs) == 1:
            return ctx.decode(seqs[0], int(tokens[0][0])) if len(tokens[0]) == 1 else ctx.prefill(seqs[0], tokens[0])
        return ctx.forward_batch([gw.Segment(s, t) for s, t in zip(seqs, tokens)])[0]
    if r != gw.RQ_OK:
        raise RuntimeError(f"{case}: code {r}")
    return state["out"]


def work(case):
    if case["kind"] != "step":
        n, k, m = case["n"], case["k"], case["m"]
        w = n * k * 34 / 32 if case["kind"] == "q8" else n * (k // 256) * KQ_BYTES[case["type"]]
        return {"bytes": w + m * k * 36 / 32 + 4 * m * n, "flops": 2 * m * n * k}
    d, wb = _shape(case["model"])
    lens, new = _lists(case)
    rows, qd, kvd = sum(new), d["n_heads"] * d["head_dim"], d["n_kv_heads"] * d["head_dim"]
    layer = d["dim"] * (2 * qd + 2 * kvd + 3 * d["hidden"])  # weights
    head = d["dim"] * d["vocab"]
    kvb = 2 * kvd * KV_BYTES[case["kv"]]
    pairs = sum(n * a + n * (n + 1) // 2 for a, n in zip(lens, new))
    b = d["n_layers"] * (layer * wb + kvb * (sum(lens) + rows)) + head * wb + 4 * len(new) * d["vocab"]
    f = 2 * rows * layer * d["n_layers"] + 2 * len(new) * head + 4 * d["n_layers"] * qd * pairs
    return {"bytes": b, "flops": f}


def tolerance(case):
    return "exact"


# ------------------------------------------------------------------------------------------------- 64-bit results

def _q4k(b, five):
    """Q4_K / Q5_K super-blocks (uint8 [nblk, 144 / 176]) -> [nblk, 256] values."""
    d = b[:, :4].contiguous().view(torch.float16).double()
    s = b[:, 4:16].long()
    sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | (s[:, :4] >> 6) << 4], 1)
    mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | (s[:, 4:8] >> 6) << 4], 1)
    q = b[:, -128:].long().reshape(-1, 4, 1, 32)
    q = torch.cat([q & 15, q >> 4], 2).reshape(-1, 8, 32)
    if five:
        q = q | ((b[:, 16:48].long()[:, None, :] >> torch.arange(8, device=b.device)[None, :, None]) & 1) << 4
    return (d[:, :1, None] * sc[..., None] * q - d[:, 1:, None] * mn[..., None]).reshape(-1, 256)


def _q6k(b):
    lo, hi = b[:, :128].long().reshape(-1, 2, 1, 2, 32), b[:, 128:192].long().reshape(-1, 2, 1, 32)
    low = torch.cat([lo & 15, lo >> 4], 2).reshape(-1, 2, 4, 32)
    top = torch.cat([(hi >> (2 * p)) & 3 for p in range(4)], 2)
    q = ((low | top << 4) - 32).reshape(-1, 16, 16)
    sc = b[:, 192:208].contiguous().view(torch.int8).double()
    return (b[:, 208:210].contiguous().view(torch.float16).double()[:, :, None] * sc[..., None] * q).reshape(-1, 256)


def _q8(b):
    return b[:, :2].contiguous().view(torch.float16).double() * b[:, 2:].contiguous().view(torch.int8).double()


def _gguf(path):
    """The tensors of a GGUF file as (type, numpy bytes, dims); metadata read over."""
    raw = np.memmap(path, np.uint8, "r")
    at = 24
    fixed = {0: 1, 1: 1, 2: 2, 3: 2, 4: 4, 5: 4, 6: 4, 7: 1, 10: 8, 11: 8, 12: 8}

    def u(size):
        nonlocal at
        at += size
        return int.from_bytes(raw[at - size:at].tobytes(), "little")

    def text():
        nonlocal at
        n = u(8)
        at += n
        return raw[at - n:at].tobytes().decode()

    def skip(t):
        nonlocal at
        if t == 8:
            text()
        elif t == 9:
            et, n = u(4), u(8)
            if et in fixed:
                at += n * fixed[et]
            else:
                for _ in range(n):
                    skip(et)
        else:
            at += fixed[t]

    n_tensors, n_meta = (int.from_bytes(raw[o:o + 8].tobytes(), "little") for o in (8, 16))
    for _ in range(n_meta):
        text()
        skip(u(4))
    info = []
    for _ in range(n_tensors):
        name = text()
        dims = [u(8) for _ in range(u(4))]
        info.append((name, dims, u(4), u(8)))
    data = (at + 31) // 32 * 32
    size = {0: (1, 4), 8: (32, 34), 12: (256, 144), 14: (256, 210)}
    return {name: (t, raw[data + o:data + o + math.prod(dims) // size[t][0] * size[t][1]], dims) for name, dims, t, o in info}


def _tensor(g, name):
    t, raw, dims = g[name]
    b = torch.from_numpy(np.array(raw)).to(DEV)
    if t == 0:
        return b.view(torch.float32).double()
    b = b.reshape(-1, {8: 34, 12: 144, 14: 210}[t])
    v = _q8(b) if t == 8 else _q4k(b, False) if t == 12 else _q6k(b)
    return v.reshape(dims[1], dims[0])


def _quantized(x):
    g = x.reshape(x.shape[0], -1, 32)
    top = g.abs().amax(-1, keepdim=True)
    y = g * torch.where(top > 0, 127 / top, top)
    return (torch.trunc(y + torch.copysign(torch.full_like(y, 0.49999997), y)) * (top / 127)).reshape(x.shape)


def _norm(x, w):
    return w * x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-6)


def _synthetic_kv(seed, layer, n, d):
    """rq_seq_fill_synthetic's f16 caches as [n, kv heads, head_dim] (its element order: blocks of 256 positions, heads; K
    in tiles of 16 positions transposed, V in rows)."""
    nb, h, e = (n + 255) // 256, d["n_kv_heads"], d["head_dim"]

    def wrap(v):
        return (v + (1 << 63)) % (1 << 64) - (1 << 63)

    def shr(z, s):
        return (z >> s) & ((1 << (64 - s)) - 1)

    z = torch.arange(nb * 256 * h * e, device=DEV) * wrap(0x9e3779b97f4a7c15) + wrap(seed + layer * 0x1000193)
    z = (z ^ shr(z, 30)) * wrap(0xbf58476d1ce4e5b9)
    z = (z ^ shr(z, 27)) * wrap(0x94d049bb133111eb)
    z = z ^ shr(z, 31)
    a, b = ((z >> o & 0xffffff).float() * (1 / 16777216) for o in (0, 24))
    k = ((2 * a - 1) * 3.9).half().reshape(nb, h, 16, e, 16).permute(0, 2, 4, 1, 3).reshape(-1, h, e)
    v = ((2 * b - 1) * 0.99).half().reshape(nb, h, 256, e).permute(0, 2, 1, 3).reshape(-1, h, e)
    return k[:n].double(), v[:n].double()


def _attend(q, k, v, pos):
    """Causal attention of rows q [n, heads, e] at positions pos over k, v [len, kv heads, e]."""
    n, heads, e = q.shape
    kvh = k.shape[1]
    qg = q.reshape(n, kvh, heads // kvh, e).permute(1, 0, 2, 3).reshape(kvh, -1, e)
    s = torch.matmul(qg, k.permute(1, 2, 0).contiguous()) / math.sqrt(e)
    dead = torch.arange(k.shape[0], device=DEV)[None, :] > pos.repeat_interleave(heads // kvh)[:, None]
    p = torch.softmax(s.masked_fill(dead, float("-inf")), -1)
    o = torch.matmul(p, v.permute(1, 0, 2).contiguous())
    return o.reshape(kvh, n, heads // kvh, e).permute(1, 0, 2, 3).reshape(n, heads * e)


def _model_exact(case, seed):
    lens, new = _lists(case)
    d, _ = _shape(case["model"])
    with tempfile.TemporaryDirectory() as tmp:
        g = _gguf(_write(case["model"], tmp))
        tok = torch.from_numpy(_tokens(seed, d["vocab"], sum(lens) + sum(new)).astype(np.int64)).to(DEV)
        prompt = case["fill"] == "prompt"
        ids, pos, start, cut, o = [], [], [], [], 0
        for have, n in zip(lens, new):
            first = 0 if prompt else have
            ids.append(tok[o + first:o + have + n])
            pos.append(torch.arange(first, have + n, device=DEV))
            start.append(first)
            cut.append(have + n - first)
            o += have + n
        ids, allpos = torch.cat(ids), torch.cat(pos)
        e, qh, kh, half = d["head_dim"], d["n_heads"], d["n_kv_heads"], d["head_dim"] // 2
        theta = d.get("rope_theta", 0) or 1e6
        ang = allpos[:, None, None].double() * theta ** (-torch.arange(half, device=DEV).double() / half)
        cos, sin = torch.cos(ang), torch.sin(ang)

        def rope(x):
            a, b = x[..., :half], x[..., half:]
            return torch.cat([a * cos - b * sin, a * sin + b * cos], -1)

        x = _tensor(g, "token_embd.weight")[ids]
        for layer in range(d["n_layers"]):
            def w(name):
                return _tensor(g, f"blk.{layer}.{name}.weight")

            def mm(x, name):
                return torch.matmul(x, w(name).t().contiguous())

            h = _quantized(_norm(x, w("attn_norm")))
            q, k, v = (mm(h, f"attn_{c}").reshape(len(ids), -1, e) for c in "qkv")
            q, k = rope(_norm(q, w("attn_q_norm"))), rope(_norm(k, w("attn_k_norm"))).half().double()
            v, att, r = v.half().double(), [], 0
            for i, (n, first, p) in enumerate(zip(cut, start, pos)):
                ks, vs = k[r:r + n], v[r:r + n]
                if first:
                    k0, v0 = _synthetic_kv(_fill_seed(seed, i), layer, first, d)
                    ks, vs = torch.cat([k0, ks]), torch.cat([v0, vs])
                att.append(torch.cat([_attend(q[r + c:r + min(c + 64, n)], ks, vs, p[c:c + 64]) for c in range(0, n, 64)]))
                r += n
            x = x + mm(_quantized(torch.cat(att)), "attn_output")
            h = _quantized(_norm(x, w("ffn_norm")))
            x = x + mm(_quantized(torch.nn.functional.silu(mm(h, "ffn_gate")) * mm(h, "ffn_up")), "ffn_down")
        last = torch.cumsum(torch.tensor(cut), 0).to(DEV) - 1
        h = _quantized(_norm(x[last], _tensor(g, "output_norm.weight")))
        out = torch.matmul(h, _tensor(g, "output.weight" if "output.weight" in g else "token_embd.weight").t().contiguous())
    out = out.cpu().numpy()
    return out[0] if len(lens) == 1 else out


def exact(case, seed):
    if case["kind"] == "step":
        # (the q8 and bf16 caches store other values in other orders; a chunked prompt is one causal pass here)
        return _model_exact(case, seed) if case["kv"] == "f16" else None
    s = _op_inputs(case, seed)
    n, k, m = case["n"], case["k"], case["m"]
    x = (s["xq"].double().reshape(m, -1, 32) * s["xs"].double()[..., None]).reshape(m, k)
    if case["kind"] == "q8":
        w = (s["codes"].double().reshape(n, -1, 32) * s["scales"].double()[..., None]).reshape(n, k)
    else:
        w = _q4k(s["blocks"], case["type"] == Q5_K).reshape(n, k)
    return torch.matmul(x, w.t().contiguous())
