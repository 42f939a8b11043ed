"""Performance cases: the work a user of this package has it do, one dict per case.

Every case runs the package's public Python entry points (bpd_substrate_amd.gpu's tensor
helpers, llama.DecodeModel, llama.Forward) on seeded random tensors in GGUF block formats.
Kinds of case:

  dequant      Q4_K -> fp32 of a whole tensor (loading a model, inspecting weights)
  q4k, q6k     one token's product with one matrix of each of `layers` layers
  q4k_chain    the same in the reference CPU's sequential fp32 order (parity checks)
  q8_0         Q8_0 matrix x 1..512 activation rows, in either reference order: one row is a
               decode step, a few rows a batch of users or drafted tokens, many rows a prefill
  decode       one token through a whole model (llama.DecodeModel)
  forward      several tokens through a whole model (llama.Forward)

`layers` > 1 gives a call the cold weights that a model's layers have.  Quants are uniform,
scales half-normal, sized so that weights have a standard deviation of about 0.02 and the
activations stay near N(0, 1), as in a trained model.
"""
import numpy as np
import torch

from bpd_substrate_amd import formats, gpu, llama

MATS = llama.MATRICES


# ---------------------------------------------------------------- the cases

def listed():
    return [
        # the smallest call: a K or V projection of a 2048-wide model, one token; latency counts
        dict(name="q4k_kv_1024x2048", kind="q4k", M=1024, K=2048, layers=1, x="f32", order=0),
        # the FFN up projection of a 7B-shaped layer from a Q8_K activation, four layers of it
        dict(name="q4k_up_14336x4096", kind="q4k", M=14336, K=4096, layers=4, x="q8k", order=0),
        # the output head of a Q4_K_M file
        dict(name="q6k_head_32000x4096", kind="q6k", M=32000, K=4096, layers=1),
        # a harness that compares with the reference CPU bit for bit
        dict(name="q4k_chain_14336x4096", kind="q4k_chain", M=14336, K=4096, layers=1),
        # a whole weight tensor to fp32
        dict(name="dequant_4096x4096", kind="dequant", n=4096 * 4096, order=0),
        # Q8_0 decode: the down projection of a 7B-shaped layer, one token, two layers of it
        dict(name="q8_0_down_1x4096x14336", kind="q8_0", M=4096, K=14336, tokens=1, layers=2, order="T"),
        # Q8_0 with a few rows at once: eight users, or eight drafted tokens
        dict(name="q8_0_up_8x14336x4096", kind="q8_0", M=14336, K=4096, tokens=8, layers=2, order="T"),
        # prefill of a square projection in the default order
        dict(name="q8_0_prefill_512x4096x4096", kind="q8_0", M=4096, K=4096, tokens=512, layers=1, order="T"),
        # prefill of the up projection in the scalar order
        dict(name="q8_0_prefill_s_512x14336x4096", kind="q8_0", M=14336, K=4096, tokens=512, layers=1, order="S"),
        # a long chat on a Q4_K_M model: binary16 cache, 2,048 rows of context
        dict(name="decode_q4km_ctx2048", kind="decode", fmt="q4km", L=4, E=4096, H=32, HKV=8, F=14336, V=32000,
             S=4096, pos=2047, f16=True),
        # the reference GPU driver's own loop: padded Q8 weights, one synchronous token per call
        dict(name="decode_pad8_ctx256", kind="decode", fmt="pad8", L=4, E=4096, H=32, HKV=8, F=14336, V=32000,
             S=2048, pos=255, f16=False),
        # a 512-token prompt through the multi-token forward, logits of every token; the largest
        dict(name="forward_512", kind="forward", L=2, E=4096, H=32, HKV=8, F=14336, V=32000, S=2048, T=512, kv=0,
             order="T", f16=True),
    ]


def _log(rng, lo, hi, step=1):
    """A size spread over the logarithm of [lo, hi], a multiple of `step`."""
    v = int(round(lo * (hi / lo) ** rng.random()))
    return max(-(-lo // step) * step, v // step * step)


def _shape(rng, blk):
    """A model shape: width 1024..4096, GQA groups of 1..8, FFN 2..3.5 times the width."""
    E, D = rng.choice([1024, 1536, 2048, 2560, 3072, 4096]), rng.choice([64, 128])
    H = E // D
    g = rng.choice([g for g in (1, 2, 4, 8) if H % g == 0])
    return dict(E=E, H=H, HKV=H // g, F=max(blk, int(E * rng.uniform(2.0, 3.5)) // blk * blk))


def draw(rng):
    kind = rng.choice(["dequant", "q4k", "q4k", "q6k", "q4k_chain", "q8_0", "q8_0", "q8_0", "q8_0", "decode", "decode",
                       "decode", "forward", "forward"])
    if kind == "dequant":
        return dict(kind=kind, n=256 * _log(rng, 64, 131072), order=rng.randrange(2))
    if kind == "q4k":
        x = rng.choice(["f32", "q8k"])
        return dict(kind=kind, M=_log(rng, 256, 32000), K=_log(rng, 1024, 16384, 256), layers=1, x=x,
                    order=0 if x == "f32" else rng.randrange(2))
    if kind in ("q6k", "q4k_chain"):
        return dict(kind=kind, M=_log(rng, 256, 32000 if kind == "q6k" else 14336), K=_log(rng, 1024, 14336, 256),
                    layers=1)
    if kind == "q8_0":
        tokens = rng.choice([1, _log(rng, 2, 32), _log(rng, 33, 512)])
        return dict(kind=kind, M=_log(rng, 256, 14336), K=_log(rng, 1024, 14336, rng.choice([32, 128, 1024])),
                    tokens=tokens, layers=1, order=rng.choice(["T", "T", "S"]))
    if kind == "decode":
        fmt = rng.choice(["q4k", "q4km", "pad8"])
        S = 4096
        return dict(kind=kind, fmt=fmt, L=rng.choice([1, 2, 4]), **_shape(rng, 32 if fmt == "pad8" else 256),
                    V=_log(rng, 4000, 32000, 8), S=S, pos=_log(rng, 1, S - 1), f16=fmt != "pad8" and rng.random() < 0.7)
    T = _log(rng, 1, 512)
    return dict(kind=kind, L=rng.choice([1, 2]), **_shape(rng, 32), V=_log(rng, 4000, 32000, 8), S=2048, T=T,
                kv=rng.choice([0, _log(rng, 1, 1024)]), order=rng.choice(["T", "T", "S"]), f16=rng.random() < 0.7)


# ---------------------------------------------------------------- random tensors, made on the GPU

class _Gen:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, n, sigma=1.0):
        return torch.randn(n, generator=self.g, device="cuda") * sigma

    def bytes(self, *shape):
        return torch.randint(0, 256, shape, generator=self.g, device="cuda", dtype=torch.uint8)

    def scales(self, n, sigma):
        return (self.normal(n).abs() * sigma).half()

    def norm_w(self, n):
        return 1.0 + 0.1 * self.normal(n)

    def q4k(self, rows, k):
        nb = rows * (k // 256)
        b = self.bytes(nb, 144)
        d = self.scales(nb, 8e-5)
        b[:, 0:2] = d.view(torch.uint8).reshape(nb, 2)
        b[:, 2:4] = (d * 7.5).view(torch.uint8).reshape(nb, 2)   # zero-mean weights
        return b.reshape(-1)

    def q6k(self, rows, k):
        nb = rows * (k // 256)
        b = self.bytes(nb, 210)
        b[:, 208:210] = self.scales(nb, 1.5e-5).view(torch.uint8).reshape(nb, 2)
        return b.reshape(-1)

    def q8_0_parts(self, rows, k, sigma=3e-4):
        nb = rows * (k // 32)
        q = torch.randint(-127, 128, (nb, 32), generator=self.g, device="cuda", dtype=torch.int8)
        return self.scales(nb, sigma).view(torch.uint8).reshape(nb, 2), q.view(torch.uint8)

    def q8_0(self, rows, k, sigma=3e-4):
        d, q = self.q8_0_parts(rows, k, sigma)
        return torch.cat([d, q], 1).reshape(-1)

    def pad8(self, rows, k):
        """The padded layout [k/32][rows][64] of the same values as q8_0()."""
        d, q = self.q8_0_parts(rows, k)
        out = torch.zeros(k // 32, rows, 64, device="cuda", dtype=torch.uint8)
        out[:, :, 0:2] = d.reshape(rows, k // 32, 2).transpose(0, 1)
        out[:, :, 4:36] = q.reshape(rows, k // 32, 32).transpose(0, 1)
        return out.reshape(-1)


def _dims(c):
    E, F, kv = c["E"], c["F"], c["HKV"] * (c["E"] // c["H"])
    return {"q": (E, E), "k": (kv, E), "v": (kv, E), "o": (E, E), "gate": (F, E), "up": (F, E), "down": (E, F)}


def _q4km(c, l):
    """Matrices of layer l that a Q4_K_M file keeps in Q6_K."""
    return {"v": llama.W_Q6K_GGUF, "down": llama.W_Q6K_GGUF} if c["fmt"] == "q4km" and l % 2 == 0 else {}


def _cache(g, c, rows, f16):
    """One cache of c["S"] rows, the first `rows` holding finite data."""
    row = c["HKV"] * (c["E"] // c["H"])
    t = torch.zeros(c["S"] * row, device="cuda")
    t[:rows * row] = g.normal(rows * row)
    return t.half().view(torch.int16) if f16 else t


# ---------------------------------------------------------------- prepare, run

def prepare(case, seed):
    c, g = case, _Gen(seed)
    s = dict(c)
    kind = c["kind"]
    if kind == "dequant":
        s["w"] = g.q4k(c["n"] // 256, 256)
        s["out"] = torch.empty(c["n"], device="cuda")
    elif kind in ("q4k", "q6k", "q4k_chain"):
        make = g.q6k if kind == "q6k" else g.q4k
        s["w"] = [make(c["M"], c["K"]) for _ in range(c["layers"])]
        s["a"] = [g.normal(c["K"]) for _ in range(c["layers"])]
        if kind == "q6k" or c.get("x") == "q8k":
            s["a"] = [gpu.quant_q8_k(a) for a in s["a"]]
        s["out"] = [torch.empty(c["M"], device="cuda") for _ in range(c["layers"])]
    elif kind == "q8_0":
        s["w"] = [g.q8_0(c["M"], c["K"]) for _ in range(c["layers"])]
        s["a"] = [g.normal(c["tokens"] * c["K"]) for _ in range(c["layers"])]
        s["out"] = [torch.empty(c["tokens"] * c["M"], device="cuda") for _ in range(c["layers"])]
    elif kind == "decode":
        _prepare_decode(s, c, g)
    else:
        _prepare_forward(s, c, g)
    return s


def _prepare_decode(s, c, g):
    pad8 = c["fmt"] == "pad8"
    fmt = llama.W_Q8_PAD64 if pad8 else llama.W_Q4K_GGUF
    make = {llama.W_Q8_PAD64: g.pad8, llama.W_Q4K_GGUF: g.q4k, llama.W_Q6K_GGUF: g.q6k}
    formats_l = [_q4km(c, l) for l in range(c["L"])]
    lm = llama.W_Q6K_GGUF if c["fmt"] == "q4km" else fmt
    layers = []
    for l in range(c["L"]):
        d = {"attn_norm": g.norm_w(c["E"]), "ffn_norm": g.norm_w(c["E"])}
        for m, (rows, k) in _dims(c).items():
            d[m] = make[formats_l[l].get(m, fmt)](rows, k)
        layers.append(d)
    cfg = dict(n_layers=c["L"], n_embd=c["E"], n_head=c["H"], n_head_kv=c["HKV"], head_dim=c["E"] // c["H"],
               ff_dim=c["F"], vocab_size=c["V"], max_seq=c["S"], eps=1e-5, rope_theta=10000.0)
    more = {} if pad8 else dict(formats=formats_l, lm_format=lm, kv_cache_f16=c["f16"])
    s["layers"], s["norm"], s["lm"] = layers, g.norm_w(c["E"]), make[lm](c["V"], c["E"])
    s["model"] = m = llama.DecodeModel(cfg, layers, s["norm"], lm_head=s["lm"], fmt=fmt, **more)
    for t in m.k_cache + m.v_cache:
        t.copy_(_cache(g, c, c["pos"], c["f16"]))
    s["emb"] = g.normal(c["E"])


def _prepare_forward(s, c, g):
    layers = []
    for _ in range(c["L"]):
        d = {"attn_norm_w": g.norm_w(c["E"]), "ffn_norm_w": g.norm_w(c["E"])}
        for m, (rows, k) in _dims(c).items():
            d["w_" + m] = g.q8_0(rows, k)
        layers.append(d)
    D = c["E"] // c["H"]
    cfg = dict(n_layers=c["L"], n_heads=c["H"], n_kv_heads=c["HKV"], head_dim=D, embed_dim=c["E"], ffn_dim=c["F"],
               vocab_size=c["V"], max_seq_len=c["S"], rms_eps=1e-5, rope_base=10000.0, rope_dim=D,
               kv_cache_f16=int(c["f16"]))
    s["layers"], s["embd"], s["norm"], s["lm"] = (layers, g.q8_0(c["V"], c["E"], 0.012), g.norm_w(c["E"]),
                                                  g.q8_0(c["V"], c["E"]))
    s["model"] = f = llama.Forward(cfg, layers, s["embd"], s["norm"], s["lm"])
    for t in (f.k_cache, f.v_cache):
        t.copy_(torch.cat([_cache(g, c, c["kv"], c["f16"]) for _ in range(c["L"])]))
    s["ids"] = torch.randint(0, c["V"], (c["T"],), generator=g.g, device="cuda").cpu().numpy().astype(np.int32)
    s["pos_ids"] = np.arange(c["kv"], c["kv"] + c["T"], dtype=np.int32)


def run(state):
    s = state
    kind = s["kind"]
    if kind == "dequant":
        return gpu.dequant_q4k(s["w"], s["order"], out=s["out"])
    if kind == "decode":
        return _run_decode(s)
    if kind == "forward":
        logits, toks = s["model"].forward(s["ids"], s["pos_ids"], s["kv"], order=s["order"])
        return {"logits": logits, "tokens": toks, "k": _values(s["model"].k_cache), "v": _values(s["model"].v_cache)}
    M, K = s["M"], s["K"]
    for w, a, out in zip(s["w"], s["a"], s["out"]):
        if kind == "q8_0":
            f = gpu.qmatmul_q8_0_llamafile if s["order"] == "T" else gpu.qmatmul_q8_0_llamafile_s
            f(w, a, M, s["tokens"], K, out=out)
        elif kind == "q4k_chain":
            gpu.qmatmul_q4k(w, a, M, K, out=out)
        elif kind == "q6k":
            gpu.qmatmul_q6k_q8k(w, a, M, K, order=formats.ORDER_GGUF, out=out)
        elif s["x"] == "f32":
            gpu.qmatmul_q4k_q8k_fused(w, a, M, K, out=out)
        else:
            gpu.qmatmul_q4k_q8k(w, a, M, K, order=s["order"], out=out)
    return s["out"]


def _run_decode(s):
    m = s["model"]
    token = None
    if s["fmt"] == "pad8":
        token = m.step(s["emb"], s["pos"])   # generate_token(): waits for the token
    else:
        m.enqueue(s["emb"], s["pos"])        # a serving loop: the token stays on the device
    token = m.buf_t["argmax_result"][:1] if token is None else token
    return {"logits": m.buf_t["logits"], "x": m.buf_t["x"], "token": token,
            "k": [_values(t) for t in m.k_cache], "v": [_values(t) for t in m.v_cache]}


def _values(cache):
    return cache.view(torch.float16) if cache.dtype == torch.int16 else cache


# ---------------------------------------------------------------- work and tolerance

_BPW = {"q4k": 144 / 256, "q6k": 210 / 256, "q8_0": 34 / 32, "pad8": 2}   # bytes per weight


def work(case):
    c = case
    kind = c["kind"]
    if kind == "dequant":
        return {"bytes": c["n"] * (144 / 256 + 4), "flops": 2 * c["n"]}
    if kind in ("q4k", "q6k", "q4k_chain", "q8_0"):
        T, L = c.get("tokens", 1), c["layers"]
        w = _BPW["q4k" if kind == "q4k_chain" else kind] * c["M"] * c["K"]
        a = c["K"] * (292 / 256 if kind == "q6k" or c.get("x") == "q8k" else 4)
        return {"bytes": L * (w + T * a + T * c["M"] * 4), "flops": L * 2 * c["M"] * c["K"] * T}
    T = c.get("T", 1)
    first = c["pos"] if kind == "decode" else c["kv"]
    kv_row, esz = c["HKV"] * (c["E"] // c["H"]), 2 if c["f16"] else 4
    n_w, bytes_ = 0, 0
    for l in range(c["L"]):
        q6 = _q4km(c, l) if kind == "decode" else {}
        for m, (rows, k) in _dims(c).items():
            n_w += rows * k
            bytes_ += rows * k * (_BPW["q6k"] if m in q6 else _weight_bytes(c))
    n_w += c["V"] * c["E"]
    bytes_ += c["V"] * c["E"] * (_BPW["q6k"] if c.get("fmt") == "q4km" else _weight_bytes(c))
    ctx = sum(first + t + 1 for t in range(T))
    bytes_ += 2 * c["L"] * (first + T) * kv_row * esz + T * (c["V"] + c["E"]) * 4
    return {"bytes": bytes_, "flops": 2 * n_w * T + 4 * c["L"] * c["E"] * ctx}


def _weight_bytes(c):
    return _BPW["q4k" if c.get("fmt") in ("q4k", "q4km") else c.get("fmt", "q8_0")]


def tolerance(case):
    """Dequantization is one rounding per value.  The products sum exact integers per block in
    fp32, so another order of the block sums is off by a few roundings (measured: Q4_K and Q6_K
    within 1e-7 of 64 bits, Q8_0's two orders 5.6e-7 apart at K = 14336; the sequential chain of
    fp32 products 1.2e-6 from 64 bits at K = 4096, growing with the root of K).  In a whole model
    a rounding moves some activations across a quantization step: orders T and S of one forward
    are 1.5e-2 apart in the logits after 2 layers and pick another token in 4 rows of 100."""
    kind = case["kind"]
    if kind == "dequant":
        return "exact"
    if kind == "q4k_chain":
        return {"rel": 1e-5, "max": 1e-4}
    if kind in ("q4k", "q6k", "q8_0"):
        return {"rel": 2.5e-6, "max": 1e-5}
    return {"rel": 2e-2, "max": 0.5, "differ": 0.01}


# ---------------------------------------------------------------- the same in 64 bits

def _f16(b):
    return b.contiguous().view(torch.float16).double()


def _w_q4k(raw, rows, k, order):
    b = raw.reshape(-1, 144)
    d, dmin, s, qs = _f16(b[:, 0:2]), _f16(b[:, 2:4]), b[:, 4:16].int(), b[:, 16:].int()
    sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).double()
    mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
    lo, hi = (qs & 15).double(), (qs >> 4).double()
    if order == 0:   # sub-block j: 16 low nibbles, then 16 high nibbles, of qs[16j..16j+15]
        q = torch.stack([lo.reshape(-1, 8, 16), hi.reshape(-1, 8, 16)], 2).reshape(-1, 8, 32)
    else:            # sub-blocks 2i, 2i+1: the low, the high nibbles of qs[32i..32i+31]
        q = torch.stack([lo.reshape(-1, 4, 32), hi.reshape(-1, 4, 32)], 2).reshape(-1, 8, 32)
    return ((d * sc)[:, :, None] * q - (dmin * mn)[:, :, None]).reshape(rows, k)


def _w_q6k(raw, rows, k):
    b = raw.reshape(-1, 210)
    ql, qh, sc, d = b[:, 0:128].int().reshape(-1, 2, 64), b[:, 128:192].int().reshape(-1, 2, 32), \
        b[:, 192:208].contiguous().view(torch.int8).double(), _f16(b[:, 208:210])
    parts = [(ql[:, :, 0:32] & 15) | ((qh & 3) << 4), (ql[:, :, 32:64] & 15) | (((qh >> 2) & 3) << 4),
             (ql[:, :, 0:32] >> 4) | (((qh >> 4) & 3) << 4), (ql[:, :, 32:64] >> 4) | (((qh >> 6) & 3) << 4)]
    q = torch.stack(parts, 2).reshape(-1, 16, 16).double() - 32
    return ((d * sc)[:, :, None] * q).reshape(rows, k)


def _w_q8_0(raw, rows, k):
    b = raw.reshape(-1, 34)
    return (_f16(b[:, 0:2]) * b[:, 2:34].contiguous().view(torch.int8).double()).reshape(rows, k)


def _w_pad8(raw, rows, k):
    b = raw.reshape(k // 32, rows, 64).transpose(0, 1)
    return (_f16(b[:, :, 0:2]) * b[:, :, 4:36].contiguous().view(torch.int8).double()).reshape(rows, k)


def _quantized(x, blk):
    """The values that the Q8_0 (32) or Q8_K (256) blocks of x hold, by the formats' own fp32 rule."""
    v = x.float().cpu().reshape(-1, blk)
    amax = v.abs().amax(1, keepdim=True)
    top = torch.full_like(amax, 127.0)   # a tensor: a scalar numerator would become a reciprocal
    d = amax / top
    q = torch.round(v * torch.where(amax > 0, top / amax, torch.zeros_like(amax)))
    d = d.half() if blk == 32 else d
    return (q.double() * d.double()).reshape(x.shape).to(x.device)


def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    if kind == "dequant":
        return _w_q4k(s["w"], 1, s["n"], s["order"]).reshape(-1)
    if kind in ("q4k", "q6k", "q4k_chain", "q8_0"):
        out = []
        for w, a in zip(s["w"], s["a"]):
            M, K, T = s["M"], s["K"], s.get("tokens", 1)
            W = _w_q6k(w, M, K) if kind == "q6k" else _w_q8_0(w, M, K) if kind == "q8_0" \
                else _w_q4k(w, M, K, s.get("order", 0))
            if kind == "q4k_chain":
                x = a.double()
            elif a.dtype == torch.uint8:
                b = a.reshape(-1, 292)
                x = b[:, 0:4].contiguous().view(torch.float32).double() * b[:, 4:260].contiguous().view(torch.int8)
            else:
                x = _quantized(a, 32 if kind == "q8_0" else 256)
            out.append((x.reshape(T, K) @ W.t().contiguous()).reshape(-1))
        return out
    return _exact_decode(s) if kind == "decode" else _exact_forward(s)


def _rms(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-5) * w.double()


def _rope(t, pos, D):
    """NORM pairs of t [T, heads, D] at positions pos [T]."""
    j = torch.arange(D // 2, device=t.device, dtype=torch.float64)
    ang = pos.double()[:, None, None] * (10000.0 ** (-2.0 * j / D))
    c, s = ang.cos(), ang.sin()
    a, b = t[..., 0::2], t[..., 1::2]
    return torch.stack([a * c - b * s, a * s + b * c], -1).reshape(t.shape)


def _layer(x, s, mat, norms, kc, vc, first, blk):
    """One layer over x [T, E] in 64 bits; kc, vc [S, HKV, D] are updated in place."""
    E, H, HKV = s["E"], s["H"], s["HKV"]
    D, T = E // H, x.shape[0]
    mul = lambda m, a: _quantized(a, blk) @ mat(m).t().contiguous()  # noqa: E731
    pos = torch.arange(first, first + T, device=x.device)
    h = _rms(x, norms[0])
    q = _rope(mul("q", h).reshape(T, H, D), pos, D)
    store = (lambda t: t.half().double()) if s["f16"] else (lambda t: t)
    kc[first:first + T] = store(_rope(mul("k", h).reshape(T, HKV, D), pos, D))
    vc[first:first + T] = store(mul("v", h).reshape(T, HKV, D))
    att = torch.empty(T, H, D, device=x.device, dtype=torch.float64)
    mask = torch.arange(first + T, device=x.device)[None, :] > pos[:, None]
    for i in range(H):
        k, v = kc[:first + T, i // (H // HKV)], vc[:first + T, i // (H // HKV)]
        sc = (q[:, i] @ k.t().contiguous()) / D ** 0.5
        att[:, i] = torch.softmax(sc.masked_fill(mask, float("-inf")), -1) @ v
    x = x + mul("o", att.reshape(T, E))
    h = _rms(x, norms[1])
    return x + mul("down", torch.nn.functional.silu(mul("gate", h)) * mul("up", h))


def _exact_decode(s):
    E, S, HKV = s["E"], s["S"], s["HKV"]
    pad8 = s["fmt"] == "pad8"
    blk = 32 if pad8 else 256
    m = s["model"]
    k = [_values(t).double().reshape(S, HKV, -1) for t in m.k_cache]
    v = [_values(t).double().reshape(S, HKV, -1) for t in m.v_cache]

    def weight(raw, rows, cols, q6):
        return _w_pad8(raw, rows, cols) if pad8 else _w_q6k(raw, rows, cols) if q6 else _w_q4k(raw, rows, cols, 1)

    x = s["emb"].double()[None]
    for l, lw in enumerate(s["layers"]):
        q6 = _q4km(s, l)
        x = _layer(x, s, lambda n: weight(lw[n], *_dims(s)[n], n in q6), (lw["attn_norm"], lw["ffn_norm"]), k[l], v[l],
                   s["pos"], blk)
    logits = _quantized(_rms(x, s["norm"]), blk) @ weight(s["lm"], s["V"], E, s["fmt"] == "q4km").t().contiguous()
    return {"logits": logits.reshape(-1), "x": x.reshape(-1), "token": None, "k": [t.reshape(-1) for t in k],
            "v": [t.reshape(-1) for t in v]}


def _exact_forward(s):
    E, S, HKV, L = s["E"], s["S"], s["HKV"], s["L"]
    f = s["model"]
    k = _values(f.k_cache).double().reshape(L, S, HKV, -1)
    v = _values(f.v_cache).double().reshape(L, S, HKV, -1)
    ids = torch.from_numpy(s["ids"]).long().to("cuda")
    x = _w_q8_0(s["embd"], s["V"], E)[ids]
    for l, lw in enumerate(s["layers"]):
        x = _layer(x, s, lambda n: _w_q8_0(lw["w_" + n], *_dims(s)[n]), (lw["attn_norm_w"], lw["ffn_norm_w"]), k[l],
                   v[l], s["kv"], 32)
    logits = _quantized(_rms(x, s["norm"]), 32) @ _w_q8_0(s["lm"], s["V"], E).t().contiguous()
    return {"logits": logits.reshape(-1), "tokens": None, "k": k.reshape(-1), "v": v.reshape(-1)}
