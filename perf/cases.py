"""The work whose speed is measured: the quantized Wan DiT path through its public entry points.

A case is a dict of plain values; ``kind`` names the entry point:

  gemm_bf16   dit.gemm_bf16: the DiT's bf16 linears around the blocks (embeddings, time projection, head)
  linear_i8   fp8.WaveW8A8Linear: per-token / per-channel int8 linear (activation quantization + GEMM)
  linear_e4m3 fp8.WaveFp8Linear: the per-tensor e4m3 linear (amax + quantization + GEMM)
  attn        backend.attn_paged_fp8: self-attention over FP8 pages, in its three forms
  cross       backend.attn_dense_bf16: cross-attention over the dense text K/V
  kv          kv.Fp8PagePool.pack and .unpack: one chunk's K/V into FP8 pages and back
  dit         dit.QuantizedWanDiT.forward_chunk: a chunk's whole denoise pass, latent -> x0

Sizes are those of the two presets (1.3B: dim 1536, 12 heads, FFN 8960, 30 layers; 14B: dim 5120, 40 heads,
FFN 13824), the 480x832 latent geometry (60 x 104 latent, 1560 tokens per frame, chunks of 3 frames), the 512-token
text context and the 21-frame attention window.  Inputs are drawn on the GPU from the seed; activations are N(0, 1)
with 1 % of the channels 20 times larger, K and V N(0, 1) with 8 heavy-tailed (Student-t, 3 degrees) dims per head.
"""

import math

import torch

from waveforcing_amd.backend import attn_dense_bf16, attn_paged_fp8
from waveforcing_amd.block import BlockParams, QuantizedWanBlock
from waveforcing_amd.dit import DiTParams, QuantizedWanDiT, gemm_bf16
from waveforcing_amd.exchange import CleanPage, PagedExchange
from waveforcing_amd.fp8 import WaveFp8Linear, WaveW8A8Linear
from waveforcing_amd.kv import Fp8PagePool, PagedKV
from waveforcing_amd.stack import QuantizedWanStack

DEV = "cuda:0"
D = 128                  # head dim
FRAME = 1560             # tokens of one 60 x 104 latent frame
CHUNK = 3 * FRAME
DIMS = {1536: dict(heads=12, ffn=8960), 5120: dict(heads=40, ffn=13824)}
EPS = 1e-6
FORMS = {"exact": {}, "qk8": {"quantized_qk": True}, "qkpv8": {"fp8_pv": True}}
BF16, F64 = torch.bfloat16, torch.float64


def listed():
    return [
        # the time projection of one chunk's 3 frames (once per new timestep): the smallest call
        dict(name="time_projection", kind="gemm_bf16", m=3, k=1536, n=9216, silu_in=True, act=""),
        # the first text-embedding linear (once per request): GELU behind a 4096-wide contraction
        dict(name="text_embedding", kind="gemm_bf16", m=512, k=4096, n=1536, silu_in=False, act="gelu"),
        # a layer's cross-attention K (or V) of the 512 text tokens (2 per layer and request)
        dict(name="text_kv_linear", kind="linear_i8", m=512, k=1536, n=1536, gelu=False, bias=True),
        # fc_in of a 1.3B block with its GELU folded in, one chunk
        dict(name="ffn_in_1p3b", kind="linear_i8", m=CHUNK, k=1536, n=8960, gelu=True, bias=True),
        # fc_out of a 14B block, one chunk
        dict(name="ffn_out_14b", kind="linear_i8", m=CHUNK, k=13824, n=5120, gelu=False, bias=True),
        # a 1.3B projection in the reference's own per-tensor e4m3 scheme
        dict(name="linear_e4m3_1p3b", kind="linear_e4m3", m=CHUNK, k=1536, n=1536, bias=True),
        # 1.3B self-attention of a chunk over the steady-state 8-chunk context, the default backend
        dict(name="attn_exact_1p3b", kind="attn", form="exact", lq=CHUNK, n_kv=8 * CHUNK, heads=12, page=FRAME),
        # 14B self-attention of a chunk early in a stream (3 chunks of context), the fp8-PV backend
        dict(name="attn_qkpv8_14b", kind="attn", form="qkpv8", lq=CHUNK, n_kv=3 * CHUNK, heads=40, page=FRAME),
        # 1.3B self-attention with single-frame chunks over 7 frames, the quantized-QK backend
        dict(name="attn_qk8_frame", kind="attn", form="qk8", lq=FRAME, n_kv=7 * FRAME, heads=12, page=FRAME),
        # 1.3B text cross-attention of a chunk
        dict(name="cross_attn_1p3b", kind="cross", lq=CHUNK, n_kv=512, heads=12),
        # one layer's K/V of a chunk published into its pages and gathered back (the paged exchange per layer)
        dict(name="kv_chunk_1p3b", kind="kv", tokens=CHUNK, heads=12, page=FRAME),
        # the whole 1.3B forward of one chunk after 8 clean chunks, from its noisy latent to x0
        dict(name="dit_chunk_1p3b", kind="dit", dim=1536, layers=30, frames=3, h=60, w=104, clean=8, t=1000.0),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["gemm_bf16", "linear_i8", "linear_i8", "linear_e4m3", "attn", "attn", "attn", "cross", "kv", "dit"])
    dim = rng.choice([1536, 1536, 5120])
    heads, ffn = DIMS[dim]["heads"], DIMS[dim]["ffn"]
    if kind == "gemm_bf16":
        k, n, lo, hi, silu, act = rng.choice([
            (256, dim, 1, 21, False, "silu"), (dim, dim, 1, 21, False, ""), (dim, 6 * dim, 1, 21, True, ""),
            (4096, dim, 1, 512, False, "gelu"), (dim, dim, 1, 512, False, ""),
            (64, dim, 390, 3 * CHUNK, False, ""), (dim, 64, 390, 3 * CHUNK, False, "")])
        return dict(kind=kind, m=_log(rng, lo, hi), k=k, n=n, silu_in=silu, act=act)
    if kind in ("linear_i8", "linear_e4m3"):
        k, n, gelu = rng.choice([(dim, dim, False), (dim, 3 * dim, False), (dim, ffn, True), (ffn, dim, False)])
        c = dict(kind=kind, m=_log(rng, 1, 2 * CHUNK), k=k, n=n, bias=rng.random() < 0.8)
        if kind == "linear_i8":
            c["gelu"] = gelu and rng.random() < 0.5
        return c
    if kind == "attn":
        c = dict(kind=kind, form=rng.choice(sorted(FORMS)), lq=_log(rng, 48, CHUNK), n_kv=_log(rng, 48, 8 * CHUNK),
                 heads=heads, page=rng.choice([FRAME, FRAME, 390, 880]))
        # the largest listed attention bounds the work
        c["n_kv"] = max(1, min(c["n_kv"], 12 * CHUNK * 8 * CHUNK // (heads * c["lq"])))
        return c
    if kind == "cross":
        return dict(kind=kind, lq=_log(rng, 48, 2 * CHUNK), n_kv=rng.choice([512, 512, _log(rng, 1, 512)]), heads=heads)
    if kind == "kv":
        return dict(kind=kind, tokens=_log(rng, 64, 8 * CHUNK), heads=heads, page=rng.choice([FRAME, FRAME, 390, 880]))
    h, w = 2 * rng.randint(8, 30), 2 * rng.randint(8, 52)
    return dict(kind=kind, dim=1536, layers=rng.randint(1, 6), frames=rng.randint(1, 3), h=h, w=w,
                clean=rng.randint(0, 8), t=rng.choice([1000.0, 937.5, 625.0]))


# ------------------------------------------------------------------ inputs
class _Draw:
    """Tensors of one seed, in the order they are asked for."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV).manual_seed(1000003 * (int(seed) % (1 << 40)) + 17)

    def normal(self, shape, std=1.0, mean=0.0, dtype=BF16):
        return (torch.randn(shape, generator=self.g, device=DEV) * std + mean).to(dtype)

    def activations(self, m, k):
        x = torch.randn((m, k), generator=self.g, device=DEV)
        x[:, torch.randperm(k, generator=self.g, device=DEV)[:max(1, k // 100)]] *= 20.0
        return x.to(BF16)

    def kv(self, tokens, heads):
        x = torch.randn((tokens, heads, D), generator=self.g, device=DEV)
        dims = torch.rand((heads, D), generator=self.g, device=DEV).argsort(dim=1)[:, :8]
        chi2 = torch.randn((tokens, heads, 8, 3), generator=self.g, device=DEV).square().sum(-1)
        at = dims.expand(tokens, heads, 8)
        x.scatter_(2, at, x.gather(2, at) / (chi2 / 3).sqrt())
        return x.to(BF16)

    def pages(self, n, pool):
        return torch.randperm(pool, generator=self.g, device=DEV)[:n].tolist()


def _linear_inputs(case, seed):
    r = _Draw(seed)
    w = r.normal((case["n"], case["k"]), 0.02)
    b = r.normal((case["n"],), 0.01) if case.get("bias", True) else None
    return r.activations(case["m"], case["k"]), w, b


def _kv_inputs(case, seed):
    r = _Draw(seed)
    n = case.get("n_kv", case.get("tokens"))
    return r, r.kv(n, case["heads"]), r.kv(n, case["heads"])


def _block_params(r, dim, ffn):
    lin = lambda o, i: r.normal((o, i), 0.02)
    vec = lambda n=dim, std=0.01, mean=0.0: r.normal((n,), std, mean)
    p = dict(modulation=r.normal((1, 6, dim), dim ** -0.5))
    for name in ("q", "k", "v", "o", "cq", "ck", "cv", "co"):
        p[name + "_w"], p[name + "_b"] = lin(dim, dim), vec()
    for name in ("norm_q", "norm_k", "norm3_w", "cnorm_q", "cnorm_k"):
        p[name] = vec(std=0.05, mean=1.0)
    p["norm3_b"] = vec()
    p["fc_in_w"], p["fc_in_b"] = lin(ffn, dim), vec(ffn)
    p["fc_out_w"], p["fc_out_b"] = lin(dim, ffn), vec()
    return p


def _dit_params(r, dim):
    p = dict(patch_w=r.normal((dim, 16, 1, 2, 2), 0.035), head_mod=r.normal((1, 2, dim), dim ** -0.5))
    for name, o, i, std in (("text1", dim, 4096, 0.02), ("text2", dim, dim, 0.02), ("time1", dim, 256, 0.02),
                            ("time2", dim, dim, 0.02), ("proj", 6 * dim, dim, 0.016), ("head", 64, dim, 0.02)):
        p[name + "_w"], p[name + "_b"] = r.normal((o, i), std), r.normal((o,), 0.01)
    p["patch_b"] = r.normal((dim,), 0.01)
    return p


def _dit_inputs(case, seed):
    r = _Draw(seed)
    dim = case["dim"]
    heads, ffn = DIMS[dim]["heads"], DIMS[dim]["ffn"]
    T = case["frames"] * (case["h"] // 2) * (case["w"] // 2)
    outer = _dit_params(r, dim)
    text = r.normal((512, 4096))
    noisy = r.normal((1, 16, case["frames"], case["h"], case["w"]))
    clean = [(r.kv(T, heads), r.kv(T, heads)) for _ in range(case["clean"])]  # a chunk's K (un-rotated) and V
    blocks = (_block_params(r, dim, ffn) for _ in range(case["layers"]))
    return T, heads, outer, text, noisy, clean, blocks


def prepare(case, seed):
    kind = case["kind"]
    if kind == "gemm_bf16":
        x, w, b = _linear_inputs(case, seed)
        if case["silu_in"] or case["k"] in (64, 256):
            x = _Draw(seed).normal(x.shape)   # embeddings and latents, without outlier channels
        return dict(kind=kind, x=x, w=w, b=b, kw=dict(silu_in=case["silu_in"], act_out=case["act"] or None))
    if kind == "linear_i8":
        x, w, b = _linear_inputs(case, seed)
        return dict(kind="linear", x=x, layer=WaveW8A8Linear(w, b, gelu=case["gelu"]))
    if kind == "linear_e4m3":
        x, w, b = _linear_inputs(case, seed)
        return dict(kind="linear", x=x, layer=WaveFp8Linear(w, b))
    if kind == "attn":
        r, k, v = _kv_inputs(case, seed)
        n_pages = -(-case["n_kv"] // case["page"])
        pool = Fp8PagePool(n_pages + 3, case["heads"], D, case["page"], DEV)
        table = pool.page_table(r.pages(n_pages, n_pages + 3))
        pool.pack(k, v, table)
        q = r.normal((case["lq"], case["heads"], D))
        return dict(kind=kind, q=q, ctx=PagedKV(pool, table, case["n_kv"]), kw=FORMS[case["form"]])
    if kind == "cross":
        r, k, v = _kv_inputs(case, seed)
        return dict(kind=kind, q=r.normal((case["lq"], case["heads"], D)), k=k, v=v)
    if kind == "kv":
        r, k, v = _kv_inputs(case, seed)
        n_pages = -(-case["tokens"] // case["page"])
        pool = Fp8PagePool(n_pages + 3, case["heads"], D, case["page"], DEV)
        return dict(kind=kind, k=k, v=v, pool=pool, table=pool.page_table(r.pages(n_pages, n_pages + 3)))
    T, heads, outer, text, noisy, clean, blocks = _dit_inputs(case, seed)
    hp, wp = case["h"] // 2, case["w"] // 2
    ex = PagedExchange(case["layers"], heads, hp * wp, case["frames"], 21, rf_step=4, device=DEV)
    stack = QuantizedWanStack([QuantizedWanBlock(BlockParams(**p), heads, DEV) for p in blocks], ex)
    dit = QuantizedWanDiT(DiTParams(**outer), stack)
    dit.set_text(text)
    for i, (k, v) in enumerate(clean):        # the stream so far: its clean chunks in every layer's pages
        for layer in range(case["layers"]):
            slot = ex.reserve(layer)
            ex.pack(layer, slot, k, v)
            ex.append_clean(layer, CleanPage(i, slot))
    if clean:
        ex.anchor_ku = clean[0][0].unsqueeze(0).expand(case["layers"], T, heads, D).contiguous()
    s = dict(kind="dit", dit=dit, noisy=noisy, t=case["t"], chunk=case["clean"])
    for _ in range(ex.n_slots - case["clean"]):   # earlier ticks of the stream: every free slot has been used
        run(s)
    return s


# -------------------------------------------------------------------- run
def run(s):
    kind = s["kind"]
    if kind == "gemm_bf16":
        return gemm_bf16(s["x"], s["w"], s["b"], **s["kw"])
    if kind == "linear":
        return s["layer"](s["x"])[0]
    if kind == "attn":
        return attn_paged_fp8(s["q"], s["ctx"], **s["kw"])
    if kind == "cross":
        return attn_dense_bf16(s["q"], s["k"], s["v"])
    if kind == "kv":
        pool = s["pool"]
        n = s["k"].shape[0]
        pool.pack(s["k"], s["v"], s["table"])
        k, v = pool.unpack(s["table"], n)
        return dict(k=k, v=v, k_codes=pool.k_codes, v_codes=pool.v_codes, k_scales=pool.k_scales,
                    v_scales=pool.v_scales)
    return s["dit"].forward_chunk(s["noisy"], s["t"], chunk=s["chunk"])


# ------------------------------------------------------------------- work
def _context_chunks(case):
    """(working chunks behind the anchor, chunks of the whole context) of a lone denoise pass."""
    f, n = case["frames"], case["clean"]
    work = min(max(0, (21 - 2 * f) // f), max(0, n - 1))
    return work, (1 + work if n else 0) + 1


def work(case):
    kind = case["kind"]
    if kind == "gemm_bf16":
        m, k, n = case["m"], case["k"], case["n"]
        return dict(bytes=2 * (m * k + n * k + n + m * n), flops=2 * m * n * k)
    if kind in ("linear_i8", "linear_e4m3"):
        m, k, n = case["m"], case["k"], case["n"]
        return dict(bytes=2 * m * k + n * k + 2 * n + 2 * m * n + (4 * n if kind == "linear_i8" else 4),
                    flops=2 * m * n * k)
    if kind == "attn":
        lq, n, h = case["lq"], case["n_kv"], case["heads"]
        return dict(bytes=4 * lq * h * D + 2 * n * h * (D + 4), flops=4 * lq * n * h * D)
    if kind == "cross":
        lq, n, h = case["lq"], case["n_kv"], case["heads"]
        return dict(bytes=4 * lq * h * D + 4 * n * h * D, flops=4 * lq * n * h * D)
    if kind == "kv":
        rows = 2 * case["tokens"] * case["heads"]
        return dict(bytes=2 * rows * (3 * D + 4), flops=0)
    dim, L = case["dim"], case["layers"]
    ffn = DIMS[dim]["ffn"]
    T = case["frames"] * (case["h"] // 2) * (case["w"] // 2)
    n_kv = _context_chunks(case)[1] * T
    weights = 6 * dim * dim + 2 * dim * ffn
    flops = L * (2 * T * weights + 4 * T * (n_kv + 512) * dim) + 4 * T * 64 * dim
    return dict(bytes=L * (weights + 2 * n_kv * dim * (D + 4) // D + 4 * 512 * dim) + 4 * 16 * 4 * T, flops=flops)


def tolerance(case):
    """About four times what the path shows against ``exact`` (bf16 results: half an ulp is 1.7e-3 in the
    2-norm).  The KV codes, scales and gathered values are the same bits in any correct implementation."""
    kind = case["kind"]
    if kind == "kv":
        return "exact"
    if kind == "attn":
        return {"rel": {"exact": 1e-2, "qk8": 1e-2, "qkpv8": 3e-2}[case["form"]]}
    if kind == "dit":
        return {"rel": 2e-2}
    return {"rel": 8e-3}


# ------------------------------------------------ the same in 64 bits
def _gelu(x):
    return 0.5 * x * (1 + torch.tanh(math.sqrt(2 / math.pi) * (x + 0.044715 * x ** 3)))


def _silu(x):
    return x * torch.sigmoid(x)


def _rows_i8(x):
    """(integer codes, scales) of the rows of x, the scale in fp32, in 64 bits."""
    s = (x.abs().amax(dim=1).float() / 127).clamp(min=1e-8)
    q = torch.round((x.float() / s[:, None]).double()).clamp(-127, 127)
    return q, s.double()


def _linear_i8(x, wq, ws, b):
    """x [M, K] in 64 bits through int8 weights; the activation codes are those of x."""
    q, s = _rows_i8(x)
    y = (q @ wq.t()) * s[:, None] * ws[None, :]
    return y if b is None else y + b.double()


def _kv_rows(x):
    """K or V [T, H, D] after its FP8 pages, in 64 bits (codes times scales), and the fp32 scales [T, H]."""
    s = (x.to(BF16).abs().amax(dim=-1) / 448).clamp(min=1e-8).float()
    c = (x.to(BF16).float() / s[..., None]).clamp(-448, 448).to(torch.float8_e4m3fn)
    return c.double() * s[..., None].double(), s


def _quantized_queries(q):
    """q after its per-row e4m3 quantization with a power-of-two scale (the quantized-QK forms)."""
    amax = q.abs().amax(dim=-1, keepdim=True)
    mant, e = torch.frexp(amax)
    e = torch.where(mant <= 0.875, e - 9, e - 8)
    e = torch.where(amax > 0, e, torch.zeros_like(e)).clamp(-127, 127)
    s = torch.ldexp(torch.ones_like(amax), e)
    return (q / s).float().clamp(-448, 448).to(torch.float8_e4m3fn).double() * s


def _attend(q, k, v):
    """softmax(q k^T / sqrt(D)) v per head; q [Lq, H, D], k and v [Lk, H, D], all in 64 bits."""
    out = torch.empty_like(q)
    for h in range(q.shape[1]):
        kt, vh = k[:, h].t().contiguous(), v[:, h].contiguous()
        for i in range(0, q.shape[0], 2048):
            s = (q[i:i + 2048, h].contiguous() @ kt) * (1 / math.sqrt(D))
            out[i:i + 2048, h] = torch.softmax(s, dim=-1) @ vh
    return out


def _norm(x):
    return (x - x.mean(-1, keepdim=True)) / torch.sqrt(x.var(-1, unbiased=False, keepdim=True) + EPS)


def _rms(x, w):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _rotate(x, frames, hp, wp, start):
    """3-D RoPE of x [T, H, D] in 64 bits: the head's 64 pairs split 22 / 21 / 21 over frame, height, width."""
    def freq(n):
        return 10000.0 ** (-torch.arange(n, dtype=F64, device=DEV) / n)
    grid = torch.meshgrid(torch.arange(start, start + frames, dtype=F64, device=DEV),
                          torch.arange(hp, dtype=F64, device=DEV), torch.arange(wp, dtype=F64, device=DEV),
                          indexing="ij")
    a = torch.cat([g.reshape(-1, 1) * freq(n) for g, n in zip(grid, (22, 21, 21))], dim=1)[:, None, :]
    x0, x1 = x[..., 0::2], x[..., 1::2]
    return torch.stack([x0 * a.cos() - x1 * a.sin(), x0 * a.sin() + x1 * a.cos()], dim=-1).flatten(2)


def _exact_dit(case, seed):
    T, heads, outer, text, noisy, clean, blocks = _dit_inputs(case, seed)
    dim, frames, hp, wp = case["dim"], case["frames"], case["h"] // 2, case["w"] // 2
    p = {k: v.double() for k, v in outer.items()}
    lin = lambda x, name: x @ p[name + "_w"].t() + p[name + "_b"]
    ctx_text = lin(_gelu(lin(text.double(), "text1")), "text2")
    ang = case["t"] * 10000.0 ** (-torch.arange(128, dtype=F64, device=DEV) / 128)
    e = lin(_silu(lin(torch.cat([ang.cos(), ang.sin()]).to(BF16).double()[None], "time1")), "time2")   # [1, dim]
    e0 = lin(_silu(e), "proj").view(6, dim)
    z = noisy.double()[0].view(16, frames, hp, 2, wp, 2).permute(1, 2, 4, 0, 3, 5).reshape(T, 64)
    x = z @ p["patch_w"].reshape(dim, 64).t() + p["patch_b"]
    work, _ = _context_chunks(case)
    start = case["clean"] * frames
    pages = []   # the clean chunks of the context: the anchor rotated for this pass, then the working set
    if clean:
        pages.append((_kv_rows(_rotate(clean[0][0].double(), frames, hp, wp, start - work * frames - frames))[0],
                      _kv_rows(clean[0][1])[0]))
        pages += [(_kv_rows(k)[0], _kv_rows(v)[0]) for k, v in clean[len(clean) - work:]] if work else []
    heads_of = lambda t: t.view(-1, heads, D)
    for b in blocks:
        qw = {n: _rows_i8(b[n + "_w"].double()) for n in ("q", "k", "v", "o", "cq", "ck", "cv", "co", "fc_in", "fc_out")}
        il = lambda t, n: _linear_i8(t, *qw[n], b[n + "_b"])
        m = b["modulation"][0].double() + e0
        a = _norm(x) * (1 + m[1]) + m[0]
        q = _rotate(heads_of(_rms(il(a, "q"), b["norm_q"])), frames, hp, wp, start)
        k = _rotate(heads_of(_rms(il(a, "k"), b["norm_k"])), frames, hp, wp, start)
        own = (_kv_rows(k)[0], _kv_rows(heads_of(il(a, "v")))[0])
        y = _attend(q, *(torch.cat([c[i] for c in pages + [own]]) for i in range(2))).reshape(T, dim)
        x = x + il(y, "o") * m[2]
        c = heads_of(_rms(il(_norm(x) * b["norm3_w"].double() + b["norm3_b"].double(), "cq"), b["cnorm_q"]))
        y = _attend(c, heads_of(_rms(il(ctx_text, "ck"), b["cnorm_k"])), heads_of(il(ctx_text, "cv"))).reshape(T, dim)
        x = x + il(y, "co")
        f = _gelu(il(_norm(x) * (1 + m[4]) + m[3], "fc_in"))
        x = x + il(f, "fc_out") * m[5]
    hm = p["head_mod"][0] + e
    flow = lin(_norm(x) * (1 + hm[1]) + hm[0], "head")
    flow = flow.view(frames, hp, wp, 2, 2, 16).permute(0, 5, 1, 3, 2, 4).reshape(frames, 16, 2 * hp, 2 * wp)
    # flow -> x0 at the sigma of the 1000-step shifted schedule nearest to t
    lin01 = torch.linspace(1.0, 0.0, 1001)[:-1]
    sig = 5.0 * lin01 / (1 + 4.0 * lin01)
    sigma = float(sig.double()[int(((sig * 1000).double() - case["t"]).abs().argmin())])
    return (noisy.double()[0].transpose(0, 1) - sigma * flow)[None]


def exact(case, seed):
    kind = case["kind"]
    if kind == "gemm_bf16":
        x, w, b = _linear_inputs(case, seed)
        if case["silu_in"] or case["k"] in (64, 256):
            x = _Draw(seed).normal(x.shape)
        x = x.double()
        y = (_silu(x) if case["silu_in"] else x) @ w.double().t() + b.double()
        return {"": lambda t: t, "gelu": _gelu, "silu": _silu}[case["act"]](y)
    if kind == "linear_i8":
        x, w, b = _linear_inputs(case, seed)
        y = _linear_i8(x.double(), *_rows_i8(w.double()), b)
        return _gelu(y) if case["gelu"] else y
    if kind == "linear_e4m3":
        x, w, b = _linear_inputs(case, seed)
        ws = (w.float().abs().amax() / 448).clamp(min=1e-8)
        wq = (w.float() / ws).to(torch.float8_e4m3fn).double()
        xs = (x.abs().amax() / 448).clamp(min=1e-8)            # in bf16, as the reference's tensor arithmetic
        xq = (x / xs).to(torch.float8_e4m3fn).double()
        y = (xq @ wq.t()) * (xs.double() * ws.double())
        return y if b is None else y + b.double()
    if kind == "attn":
        r, k, v = _kv_inputs(case, seed)
        n_pages = -(-case["n_kv"] // case["page"])
        r.pages(n_pages, n_pages + 3)
        q = r.normal((case["lq"], case["heads"], D)).double()
        return _attend(q if case["form"] == "exact" else _quantized_queries(q), _kv_rows(k)[0], _kv_rows(v)[0])
    if kind == "cross":
        r, k, v = _kv_inputs(case, seed)
        return _attend(r.normal((case["lq"], case["heads"], D)).double(), k.double(), v.double())
    if kind == "kv":
        _, k, v = _kv_inputs(case, seed)
        return dict(k=_kv_rows(k)[0], v=_kv_rows(v)[0], k_codes=None, v_codes=None, k_scales=None, v_scales=None)
    return _exact_dit(case, seed)
