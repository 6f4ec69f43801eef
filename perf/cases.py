"""Performance cases: the calls a user of gaje_hip makes, over the sizes they are made at.

  linear   one matvec of a layer or of the head, in each weight format (ops.*_gemv)
  rows     the bit-exact Q4_0 product of several activation rows (ops.q4_0_gemm): a
           small batch of requests, or a draft to verify
  product  the matrix-core Q4_0 product of a prompt's rows (ops.q4_0_gemm_mfma)
  moe      a top-2 mixture-of-experts SwiGLU layer (ops.moe_ffn, ops.moe_ffn_prepared)
  attention  one token's GQA attention over its KV cache (ops.attention)
  decode   greedy tokens of one sequence on a prompt's cache, then one token's logits
  prompt   a prompt through a whole model, bit-exact (prefill) or on the matrix
           cores (prefill_mfma), to its last token's logits
  batch    several requests stepping together: their prompts, then greedy tokens

Shapes are those of the presets of gaje_hip.synth (SmolLM2-135M, Qwen2-0.5B,
Qwen2.5-1.5B), of the benchmark's matvec and MoE legs, and generic ones.  Models
are random-init files of those shapes; where a case needs only some of a model's
layers or vocabulary, "blocks" and "vocab" say so.
"""
import getpass
import json
import math
import os
import struct
import sys
import tempfile

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "gaje-semantic-compression_amd"))

import gaje_hip  # noqa: E402
from gaje_hip import ops  # noqa: E402

DEV = "cuda"
# standard normal quantile midpoints: the 4-bit and 2-bit tables of the synthetic weights
Z16 = [-1.8627319, -1.3180109, -1.00999, -0.77642176, -0.57913216, -0.40225007, -0.23720211, -0.07841241,
       0.07841241, 0.23720211, 0.40225007, 0.57913216, 0.77642176, 1.00999, 1.3180109, 1.8627319]
Z4 = [-1.1503494, -0.31863936, 0.31863936, 1.1503494]


def listed():
    return [
        # the down matvec of a decode step of the 1.5B model: few rows, a long sum, a short call
        dict(name="matvec", kind="linear", format="q4_0", n=1536, k=8960, bias=False),
        # a gate-sized layer of the 0.5B model in the LUT format: the smallest call, latency and the launch
        dict(name="matvec-lut4", kind="linear", format="lut4", n=4864, k=896, bias=False),
        # the quantised head of an export with 8-bit embeddings: a stream of weights
        dict(name="head-q8", kind="linear", format="q8_0", n=151936, k=896, bias=False),
        # sixteen requests' rows through a QKV product with its bias, bit-exact per row
        dict(name="rows-16", kind="rows", m=16, n=2048, k=1536, bias=True),
        # a 512-token prompt's gate/up product of the 1.5B model
        dict(name="product-512", kind="product", m=512, n=17920, k=1536, bias=False),
        # a short, ragged prompt's down product: few rows, a long sum
        dict(name="product-77", kind="product", m=77, n=1536, k=8960, bias=False),
        # an MoE layer over prepared experts, a prompt's worth of tokens
        dict(name="moe-256", kind="moe", tokens=256, h=1536, ffn=4096, experts=8, prepared=True),
        # one token's attention over a long context (1.5B heads)
        dict(name="attention-4000", kind="attention", ctx=4000, capacity=4096, heads=12, kv=2, hd=128),
        # the 0.5B model's decode at batch 1 after a 512-token prompt
        dict(name="decode", kind="decode", model="qwen2-0.5b", blocks=24, vocab=151936, prompt=512, new=16),
        # a 512-token prompt on the matrix cores, 1.5B widths
        dict(name="prompt-mfma", kind="prompt", model="qwen2.5-1.5b", blocks=8, vocab=32768, tokens=512, exact=False),
        # a prompt fed bit-exactly, as the reference's own generation loop does
        dict(name="prompt-exact", kind="prompt", model="qwen2-0.5b", blocks=24, vocab=151936, tokens=201, exact=True),
        # sixteen requests served together, 1.5B widths
        dict(name="batch-16", kind="batch", model="qwen2.5-1.5b", blocks=8, vocab=32768, seqs=16, prompt=96, new=24),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _k32(rng, lo, hi):
    return max(1, _log(rng, lo, hi) // 32) * 32


HEADS = [(14, 2, 64), (12, 2, 128), (9, 3, 64), (16, 16, 64), (32, 8, 128)]


def draw(rng):
    kind = rng.choice(["linear", "linear", "rows", "product", "moe", "attention", "decode", "prompt", "prompt", "batch"])
    if kind == "linear":
        fmt = rng.choice(["q4_0", "q4_0", "q8_0", "lut4", "bit2", "f32"])
        k = _log(rng, 128, 8960) if fmt == "f32" else _k32(rng, 128, 8960)
        n = _log(rng, max(500, 8 * 10 ** 6 // k), min(160000, 151936 * 896 // k))
        return dict(kind=kind, format=fmt, n=n, k=k, bias=rng.random() < 0.4)
    if kind == "rows":
        return dict(kind=kind, m=_log(rng, 2, 64), n=_log(rng, 500, 20000), k=_k32(rng, 256, 8960), bias=rng.random() < 0.4)
    if kind == "product":
        m, k = _log(rng, 8, 1024), _k32(rng, 256, 8960)
        return dict(kind=kind, m=m, n=_log(rng, 500, min(20000, 512 * 17920 * 1536 // (m * k))), k=k, bias=rng.random() < 0.4)
    if kind == "moe":
        return dict(kind=kind, tokens=_log(rng, 1, 512), h=_k32(rng, 256, 2048), ffn=_k32(rng, 512, 4096),
                    experts=rng.choice([4, 8, 8, 16]) if rng.random() < 0.8 else 5, prepared=rng.random() < 0.6)
    if kind == "attention":
        h, kv, hd = rng.choice(HEADS)
        ctx = _log(rng, 64, 8192)
        return dict(kind=kind, ctx=ctx, capacity=max(1024, 1 << (ctx - 1).bit_length()), heads=h, kv=kv, hd=hd)
    model = rng.choice(["smollm2-135m", "qwen2-0.5b", "qwen2.5-1.5b"])
    base = dict(kind=kind, model=model, blocks=rng.randint(2, 8), vocab=rng.choice([16384, 32768, 49152]))
    if kind == "decode":
        return dict(base, prompt=_log(rng, 16, 700), new=_log(rng, 4, 48))
    if kind == "prompt":
        exact = rng.random() < 0.5
        return dict(base, tokens=_log(rng, 8, 300 if exact else 1000), exact=exact)
    return dict(base, seqs=rng.randint(2, 16), prompt=_log(rng, 16, 96), new=_log(rng, 8, 24))


# ------------------------------------------------------------------ inputs --
class Buf:
    """A torch tensor as the operator API takes device memory."""

    def __init__(self, t):
        self.t = t.contiguous()
        self.ptr, self.nbytes = self.t.data_ptr(), self.t.numel() * self.t.element_size()


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _normal(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device=DEV) * std


def _codes(g, n, nb):
    return torch.randint(0, 16, (n, nb, 32), generator=g, device=DEV, dtype=torch.uint8)


def _block_scale(g, n, nb):
    return 0.01 + 0.04 * torch.rand(n, nb, generator=g, device=DEV)


def _q4_blocks(g, n, k):
    """Rows of Q4_0 blocks: f16 scale, f16 min, 16 bytes of codes (low nibble first)."""
    nb = k // 32
    s, c = _block_scale(g, n, nb), _codes(g, n, nb)
    sc = (s * ((Z16[15] - Z16[0]) / 15)).half().view(torch.uint8).view(n, nb, 2)
    mn = (s * Z16[0]).half().view(torch.uint8).view(n, nb, 2)
    return torch.cat([sc, mn, c[..., 0::2] | (c[..., 1::2] << 4)], dim=2).contiguous()


def _q4_f64(blocks):
    n, nb, _ = blocks.shape
    sc = blocks[..., 0:2].contiguous().view(torch.float16).double()
    mn = blocks[..., 2:4].contiguous().view(torch.float16).double()
    q = torch.stack([blocks[..., 4:] & 15, blocks[..., 4:] >> 4], dim=-1).view(n, nb, 32).double()
    return (q * sc + mn).view(n, nb * 32)


def _q4_pack(blocks, k):
    n = blocks.shape[0]
    p = Buf(torch.empty(ops.q4_0_packed_bytes(n, k), dtype=torch.uint8, device=DEV))
    ops.q4_0_pack(Buf(blocks), p, n, k)
    return p


def _linear_inputs(c, seed):
    g, n, k, f = _gen(seed), c["n"], c["k"], c["format"]
    x = _normal(g, k)
    bias = _normal(g, n, std=0.02) if c["bias"] else None
    if f == "f32":
        return x, bias, (_normal(g, n, k, std=0.02),)
    nb = k // 32
    if f == "q4_0":
        return x, bias, (_q4_blocks(g, n, k),)
    if f == "q8_0":
        s = (0.0002 + 0.0004 * torch.rand(n, nb, generator=g, device=DEV)).half().view(torch.uint8).view(n, nb, 2)
        q = torch.randint(0, 255, (n, nb, 32), generator=g, device=DEV, dtype=torch.uint8)
        q = (q.to(torch.int16) - 127).to(torch.int8).view(torch.uint8)
        return x, bias, (torch.cat([s, q], dim=2).contiguous(),)
    s = _block_scale(g, n, nb)
    if f == "lut4":
        cd = _codes(g, n, nb)
        z = torch.tensor(Z16, device=DEV)
        return x, bias, (((cd[..., 0::2] << 4) | cd[..., 1::2]).contiguous(), (s[..., None] * z).contiguous())
    cd = torch.randint(0, 256, (n, nb, 8), generator=g, device=DEV, dtype=torch.uint8)
    return x, bias, (cd, (s[..., None] * torch.tensor(Z4, device=DEV)).contiguous())


def _linear_f64(c, w):
    f, n, k = c["format"], c["n"], c["k"]
    if f == "f32":
        return w[0].double()
    if f == "q4_0":
        return _q4_f64(w[0])
    if f == "q8_0":
        s = w[0][..., :2].contiguous().view(torch.float16).double()
        return (s * w[0][..., 2:].contiguous().view(torch.int8).double()).view(n, k)
    if f == "lut4":
        idx = torch.stack([w[0] >> 4, w[0] & 15], dim=-1).view(n, k // 32, 32).long()
    else:  # 2-bit codes, most significant first; 00 01 11 10 -> centroids 0 1 2 3
        raw = torch.stack([(w[0] >> sh) & 3 for sh in (6, 4, 2, 0)], dim=-1).view(n, k // 32, 32).long()
        idx = torch.tensor([0, 1, 3, 2], device=DEV)[raw]
    return torch.gather(w[1].double(), 2, idx).view(n, k)


def _rows_inputs(c, seed):
    g = _gen(seed)
    blocks = _q4_blocks(g, c["n"], c["k"])
    return blocks, _normal(g, c["m"], c["k"]), _normal(g, c["n"], std=0.02) if c["bias"] else None


def _moe_inputs(c, seed):
    g, h, f, e = _gen(seed), c["h"], c["ffn"], c["experts"]
    x, router = _normal(g, c["tokens"], h), _normal(g, e, h, std=0.02)
    return x, router, [_q4_blocks(g, 2 * f, h) for _ in range(e)], [_q4_blocks(g, h, f) for _ in range(e)]


def _attention_inputs(c, seed):
    g = _gen(seed)
    cache = (c["kv"], c["hd"], c["capacity"])
    return _normal(g, c["heads"], c["hd"]), _normal(g, *cache), _normal(g, *cache)


def _model_file(c):
    """The case's model, written once for a machine and kept among its temporary files."""
    d = os.path.join(tempfile.gettempdir(), "gaje_models_" + getpass.getuser())
    os.makedirs(d, exist_ok=True)
    path = os.path.join(d, "%s_%d_%d.flat" % (c["model"], c["blocks"], c["vocab"]))
    if not os.path.exists(path):
        part = "%s.%d" % (path, os.getpid())
        gaje_hip.synth.write_flat(part, c["model"], n_blocks=c["blocks"], vocab_size=c["vocab"], seed=3)
        os.replace(part, path)
    return path


def _tokens(c, seed, *shape):
    return np.random.default_rng(seed).integers(0, c["vocab"], shape).astype(np.uint32)


def _model_tokens(c, seed):
    if c["kind"] == "decode":
        return _tokens(c, seed, c["prompt"] + 1)
    if c["kind"] == "prompt":
        return _tokens(c, seed, c["tokens"])
    return _tokens(c, seed, c["seqs"], c["prompt"])


def _empty(*shape, dtype=torch.float32):
    return torch.empty(*shape, dtype=dtype, device=DEV)


def prepare(case, seed):
    c, s = case, {"case": case}
    kind = c["kind"]
    if kind == "linear":
        x, bias, w = _linear_inputs(c, seed)
        s["x"], s["y"], s["bias"] = Buf(x), Buf(_empty(c["n"])), Buf(bias) if c["bias"] else None
        if c["format"] == "q4_0":
            s["w"] = _q4_pack(w[0], c["k"])
        elif c["format"] == "q8_0":
            s["w"] = ops.q8_0_upload(w[0].cpu().numpy().reshape(-1), c["n"], c["k"])
        else:
            s["w"] = Buf(w[0])
            if len(w) > 1:
                s["table"], s["table_len"] = Buf(w[1]), w[1].numel()
    elif kind in ("rows", "product"):
        blocks, x, bias = _rows_inputs(c, seed)
        s["w"], s["x"], s["y"] = _q4_pack(blocks, c["k"]), Buf(x), Buf(_empty(c["m"], c["n"]))
        s["bias"] = Buf(bias) if c["bias"] else None
        if kind == "product":
            s["workspace"] = Buf(_empty(ops.q4_0_gemm_mfma_workspace(c["m"], c["n"], c["k"]), dtype=torch.uint8))
    elif kind == "moe":
        x, router, gu, dn = _moe_inputs(c, seed)
        T, h, f, e = c["tokens"], c["h"], c["ffn"], c["experts"]
        s.update(x=Buf(x), router=Buf(router), y=Buf(_empty(T, h)), idx=Buf(_empty(T, 2, dtype=torch.int32)),
                 weight=Buf(_empty(T, 2)))
        gu, dn = [_q4_pack(b, h) for b in gu], [_q4_pack(b, f) for b in dn]
        if c["prepared"]:
            s["prepared"] = Buf(_empty(ops.moe_prepared_bytes(h, f, e), dtype=torch.uint8))
            ops.moe_prepare(gu, dn, h, f, s["prepared"])
            s["workspace"] = Buf(_empty(ops.moe_ffn_prepared_workspace(T, h, f, e), dtype=torch.uint8))
        else:
            s["gate_up"], s["down"] = gu, dn
            s["workspace"] = Buf(_empty(ops.moe_ffn_workspace(T, h, f, e), dtype=torch.uint8))
    elif kind == "attention":
        q, k, v = _attention_inputs(c, seed)
        s.update(q=Buf(q), k=Buf(k), v=Buf(v), out=Buf(_empty(c["heads"], c["hd"])))
    else:
        m = gaje_hip.load_genomic_auto(_model_file(c))
        m.set_k_wta_ratio(0.0)
        s["model"], s["ids"] = m, _model_tokens(c, seed)
        if kind == "decode":
            m.reserve(c["prompt"] + c["new"] + 1)
            m.prefill(s["ids"][:-1])
        elif kind == "prompt":
            m.reserve(c["tokens"])
        else:
            s["batch"] = gaje_hip.GenomicBatch(m, c["seqs"], c["prompt"] + c["new"] + 1)
    torch.cuda.synchronize()
    return s


def run(state):
    s, c = state, state["case"]
    kind = c["kind"]
    if kind == "linear":
        n, k, nb = c["n"], c["k"], c["n"] if c["bias"] else 0
        f = c["format"]
        if f == "q4_0":
            ops.q4_0_gemv(s["w"], s["x"], s["y"], n, k, s["bias"], nb)
        elif f == "q8_0":
            ops.q8_0_gemv(s["w"], s["x"], s["y"], n, k, s["bias"], nb)
        elif f == "f32":
            ops.f32_gemv(s["w"], s["x"], s["y"], n, k, s["bias"], nb)
        elif f == "lut4":
            ops.lut4_gemv(s["w"], s["table"], s["table_len"], s["x"], s["y"], n, k, s["bias"], nb)
        else:
            ops.bit2_gemv(s["w"], s["table"], s["table_len"], s["x"], s["y"], n, k, None, s["bias"], nb)
        return s["y"].t
    if kind == "rows":
        ops.q4_0_gemm(s["w"], s["x"], s["y"], c["m"], c["n"], c["k"], s["bias"], c["n"] if c["bias"] else 0)
        return s["y"].t
    if kind == "product":
        ops.q4_0_gemm_mfma(s["w"], s["x"], s["y"], c["m"], c["n"], c["k"], s["workspace"], s["bias"],
                           c["n"] if c["bias"] else 0)
        return s["y"].t
    if kind == "moe":
        if c["prepared"]:
            ops.moe_ffn_prepared(s["x"], c["tokens"], c["h"], s["router"], c["experts"], s["prepared"], c["ffn"], s["y"],
                                 s["workspace"], s["idx"], s["weight"])
        else:
            ops.moe_ffn(s["x"], c["tokens"], c["h"], s["router"], s["gate_up"], s["down"], c["ffn"], s["y"],
                        s["workspace"], s["idx"], s["weight"])
        return {"y": s["y"].t, "experts": s["idx"].t, "weights": s["weight"].t}
    if kind == "attention":
        ops.attention(s["q"], s["k"], s["v"], c["ctx"], c["capacity"], c["heads"], c["kv"], c["hd"], s["out"])
        return s["out"].t
    m = s["model"]
    if kind == "decode":
        m.truncate_cache(c["prompt"])
        tokens = m.decode_greedy(int(s["ids"][-1]), c["new"] - 1)
        return {"tokens": tokens, "logits": m.forward(int(tokens[-1]))}
    if kind == "prompt":
        m.clear_cache_py()
        return m.prefill(s["ids"], want_logits=True) if c["exact"] else m.prefill_mfma(s["ids"], want_logits=True)
    b = s["batch"]
    b.reset()
    logits = b.feed(s["ids"], want_logits=True)
    tokens = b.decode_greedy(np.argmax(logits, axis=1).astype(np.uint32), c["new"])
    return {"prompt": logits, "tokens": tokens, "logits": b.feed(tokens[:, -1:], want_logits=True)}


# -------------------------------------------------------------- yardsticks --
def _shape(c):
    return dict(gaje_hip.synth.PRESETS[c["model"]], n_blocks=c["blocks"], vocab_size=c["vocab"])


def work(case):
    c, kind = case, case["kind"]
    q4 = 20 / 32  # bytes of a 4-bit weight with its block's scale and min
    if kind == "linear":
        n, k = c["n"], c["k"]
        b = {"q4_0": q4, "q8_0": 34 / 32, "lut4": 80 / 32, "bit2": 24 / 32, "f32": 4}[c["format"]]
        return {"bytes": n * k * b + 4 * (k + n + (n if c["bias"] else 0)), "flops": 2 * n * k}
    if kind in ("rows", "product"):
        m, n, k = c["m"], c["n"], c["k"]
        return {"bytes": n * k * q4 + 4 * (m * k + m * n), "flops": 2 * m * n * k}
    if kind == "moe":
        T, h, f, e = c["tokens"], c["h"], c["ffn"], c["experts"]
        used = e * (1 - (1 - 2 / e) ** T)  # experts that some token takes, for even routing
        return {"bytes": used * 3 * h * f * q4 + 4 * (2 * T * h + e * h + 4 * T), "flops": 2 * T * (2 * 3 * h * f + e * h)}
    if kind == "attention":
        return {"bytes": 4 * (2 * c["kv"] * c["hd"] * c["ctx"] + 2 * c["heads"] * c["hd"]),
                "flops": 4 * c["heads"] * c["hd"] * c["ctx"]}
    p = _shape(c)
    h, hd = p["n_embd"], p["n_embd"] // p["n_head"]
    kvw = p["n_head_kv"] * hd
    body = p["n_blocks"] * (h * (h + 2 * kvw) + h * h + 3 * h * p["ffn"])
    head = h * p["vocab_size"]
    kv = p["n_blocks"] * 2 * kvw * 4  # bytes of one position
    att = p["n_blocks"] * 4 * h       # operations of one (query, position) pair
    if kind == "decode":
        t, mid = c["new"], c["prompt"] + c["new"] / 2
        return {"bytes": t * (body * q4 + 4 * head + kv * mid), "flops": t * (2 * (body + head) + att * mid)}
    if kind == "prompt":
        t = c["tokens"]
        return {"bytes": body * q4 + 4 * head + kv * t, "flops": 2 * t * body + 2 * head + att * t * t / 2}
    t, steps = c["prompt"] + c["new"], c["new"] + 1
    return {"bytes": body * q4 + steps * (body * q4 + 4 * head) + c["seqs"] * kv * (t + c["new"] * t),
            "flops": c["seqs"] * (t * 2 * body + steps * 2 * head + att * t * t / 2)}


def tolerance(case):
    """About four times the distance from exact() that the paths show (a whole model's rounding grows with its depth)."""
    kind = case["kind"]
    if kind in ("linear", "rows", "product"):
        return {"rel": 2e-6}
    if kind == "moe":
        return {"rel": 4e-6, "differ": 0.002}
    if kind == "attention":
        return {"rel": 6e-6}
    return {"rel": 1e-4, "differ": 0.0}


# ------------------------------------------------------------- 64 bit path --
class _Model64:
    """The model's forward in float64 for a batch of sequences of one length: rows W x + bias, rms_norm, RoPE over
    split pairs, grouped softmax attention, SwiGLU."""

    def __init__(self, c):
        with open(_model_file(c), "rb") as f:
            head = struct.unpack_from("<4sIIIQQQQ", f.read(4096), 0)
            f.seek(4096 + head[4])
            self.dir = {e["name"]: e for e in json.loads(f.read(head[5]))}
        self.mm, self.at, self.p = np.memmap(_model_file(c), np.uint8, "r"), head[6], _shape(c)
        self.cache = [None] * c["blocks"]
        self.n = 0

    def _bytes(self, off, length):
        return torch.from_numpy(np.array(self.mm[self.at + off:self.at + off + length])).to(DEV)

    def vector(self, name):
        e = self.dir[name]
        return self._bytes(e["dna_off"], e["dna_len"]).view(torch.float32).double()

    def linear(self, name, x):
        e = self.dir[name]
        n, k = e["out_features"], e["in_features"]
        raw = self._bytes(e["dna_off"], e["dna_len"])
        w = raw.view(torch.float32).view(n, k).double() if e["bit_depth"] == 32 else _q4_f64(raw.view(n, k // 32, 20))
        y = x @ w.T
        if e["bias_len"]:
            y = y + self._bytes(e["bias_off"], e["bias_len"]).view(torch.float32).double()
        return y

    def norm(self, name, x):
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + float(np.float32(self.p["eps"]))) * self.vector(name)

    def rope(self, v, hd):
        i = torch.arange(hd // 2, device=DEV, dtype=torch.float64)
        th = torch.arange(self.n, self.n + v.shape[1], device=DEV).double()[:, None] * self.p["rope_base"] ** (-2 * i / hd)
        co, si = th.cos()[None, :, None, :], th.sin()[None, :, None, :]
        a, b = v[..., :hd // 2], v[..., hd // 2:]
        return torch.cat([a * co - b * si, a * si + b * co], dim=-1)

    def step(self, ids):
        """ids [sequences][tokens], appended to the cache; the last token's logits."""
        p = self.p
        H, KV, hd = p["n_head"], p["n_head_kv"], p["n_embd"] // p["n_head"]
        B, T = ids.shape
        e = self.dir["token_embd"]
        rows = self.mm[self.at + e["dna_off"]:self.at + e["dna_off"] + e["dna_len"]].view(np.float32).reshape(-1, p["n_embd"])
        x = torch.from_numpy(rows[ids.astype(np.int64)]).to(DEV).double()
        for i in range(p["n_blocks"]):
            b = "blk.%d." % i
            qkv = self.linear(b + "attn_qkv", self.norm(b + "attn_norm", x)).view(B, T, H + 2 * KV, hd)
            q, k, v = self.rope(qkv[:, :, :H], hd), self.rope(qkv[:, :, H:H + KV], hd), qkv[:, :, H + KV:]
            if self.cache[i] is not None:
                k, v = (torch.cat([o, n], dim=1) for o, n in zip(self.cache[i], (k, v)))
            self.cache[i] = (k, v)
            q = q.view(B, T, KV, H // KV, hd).permute(0, 2, 3, 1, 4).reshape(B * KV, -1, hd)
            ks, vs = (t.permute(0, 2, 1, 3).reshape(B * KV, -1, hd) for t in (k, v))
            s = (torch.bmm(q, ks.transpose(1, 2).contiguous()) / math.sqrt(hd)).view(B * KV, H // KV, T, -1)
            late = torch.arange(s.shape[-1], device=DEV)[None, :] > torch.arange(self.n, self.n + T, device=DEV)[:, None]
            s = s.masked_fill(late, -math.inf).softmax(-1).view(B * KV, -1, s.shape[-1])
            o = torch.bmm(s, vs).view(B, KV, H // KV, T, hd).permute(0, 3, 1, 2, 4).reshape(B, T, H * hd)
            x = x + self.linear(b + "attn_output", o)
            gu = self.linear(b + "ffn_gate_up", self.norm(b + "ffn_norm", x))
            g, u = gu.chunk(2, dim=-1)
            x = x + self.linear(b + "ffn_down", g * torch.sigmoid(g.clamp(-64, 64)) * u)
        self.n += T
        return self.linear("lm_head", self.norm("output_norm", x[:, -1]))


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "linear":
        x, bias, w = _linear_inputs(c, seed)
        y = _linear_f64(c, w) @ x.double()
        return y + bias.double() if c["bias"] else y
    if kind in ("rows", "product"):
        blocks, x, bias = _rows_inputs(c, seed)
        y = x.double() @ _q4_f64(blocks).T
        return y + bias.double() if c["bias"] else y
    if kind == "moe":
        x, router, gu, dn = _moe_inputs(c, seed)
        x = x.double()
        p, idx = (x @ router.double().T).softmax(-1).sort(dim=-1, descending=True, stable=True)
        p, idx = p[:, :2], idx[:, :2]
        weight = p / p.sum(-1, keepdim=True)
        y = torch.zeros_like(x)
        for e in range(c["experts"]):
            t, which = (idx == e).nonzero(as_tuple=True)
            g, u = (x[t] @ _q4_f64(gu[e]).T).chunk(2, dim=-1)
            y.index_add_(0, t, weight[t, which][:, None] * ((g * torch.sigmoid(g) * u) @ _q4_f64(dn[e]).T))
        return {"y": y, "experts": None, "weights": weight}
    if kind == "attention":
        q, k, v = (t.double() for t in _attention_inputs(c, seed))
        q = q.view(c["kv"], -1, c["hd"])
        w = (torch.bmm(q, k[..., :c["ctx"]].contiguous()) / math.sqrt(c["hd"])).softmax(-1)
        return torch.bmm(w, v[..., :c["ctx"]].transpose(1, 2).contiguous()).view(c["heads"], c["hd"])
    ids = _model_tokens(c, seed)
    m = _Model64(c)
    if kind == "prompt":
        return m.step(ids[None])[0]
    if kind == "decode":
        logits = m.step(ids[None])
        for _ in range(c["new"] - 1):
            logits = m.step(logits.argmax(-1).cpu().numpy()[:, None])
        return {"tokens": None, "logits": logits[0]}
    prompt = logits = m.step(ids)
    for _ in range(c["new"] + 1):
        logits = m.step(logits.argmax(-1).cpu().numpy()[:, None])
    return {"prompt": prompt, "tokens": None, "logits": logits}
