"""The work a user of libh3attn has it do, as cases to time and to check: each `kind` below is one
route through the package's public calls, as the DiT's attention block makes them.

  short    Stack.attend below 4,096 tokens (token-major operands), on post-RoPE f16 q, k, v; with
           `rope` the RMSNorm + RoPE kernel in front of it, with `smooth` K-mean smoothing
  fused    Stack.attend_fused on the fused QKV projection (4,096 tokens and up), f16 or bf16, with
           or without K-mean smoothing
  compact  the INT8 QKV projection, then Stack.attend_compact on its output
  cross    text cross-attention: the video's queries quantized, then GQA attention over the text
           keys (kept from the prompt) with a key-padding mask
  project  a hidden state quantized (prepare_plain_i8) and projected to Q, K and V^T by the INT8
           GEMM
  vsa      the block-sparse runtime (Vsa.attend), INT8 or f16 attention, with or without a gate
  int4     the INT4 operands of Q and K and the attention over them: the FP6 form, the widened
           form with a lent workspace, or its tile-skipping twin
"""
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "h3-hrx_amd"))
import h3attn as H  # noqa: E402

DEV = "cuda"
F16, BF16, F32 = "f16", "bf16", "f32"
DTYPES = {F16: torch.float16, BF16: torch.bfloat16, F32: torch.float32}
ELEMS = {F16: H.H3_ELEM_F16, BF16: H.H3_ELEM_BF16, F32: H.H3_ELEM_F32}
EPS = 1e-5


def listed():
    return [
        # a text-sized sequence at the model's 56 heads: launches and latency only
        {"name": "tiny_129", "kind": "short", "tokens": 129, "heads": 56, "smooth": False,
         "rope": False},
        # 1,024 tokens of 8 heads, the smallest benchmark configuration
        {"name": "short_1024", "kind": "short", "tokens": 1024, "heads": 8, "smooth": False,
         "rope": False},
        # an image-sized sequence on the separate route with everything it can have: RMSNorm and
        # RoPE, K-mean smoothing, an odd length
        {"name": "short_rope_smooth_2501", "kind": "short", "tokens": 2501, "heads": 56,
         "smooth": True, "rope": True},
        # just past the route's 4,096-token bound and one past a tile edge, 56 heads
        {"name": "fused_4097", "kind": "fused", "tokens": 4097, "heads": 56, "elem": F16,
         "smooth": False},
        # the 31,104-token video configuration with K-mean smoothing
        {"name": "fused_smooth_31104", "kind": "fused", "tokens": 31104, "heads": 32,
         "elem": BF16, "smooth": True},
        # the headline step: 129,024 tokens, 32 heads
        {"name": "fused_129024", "kind": "fused", "tokens": 129024, "heads": 32, "elem": BF16,
         "smooth": False},
        # video and audio queries over 512 text keys, 20 % of them padding, 32 heads over 8
        {"name": "cross_130272", "kind": "cross", "tokens": 130272, "heads": 32, "kv_heads": 8,
         "kv_tokens": 512, "pad": 0.2},
        # the projection of a text-sized f32 hidden state
        {"name": "project_513", "kind": "project", "tokens": 513, "k": 4096, "heads": 32,
         "elem": F32},
        # the projection of a video's f16 hidden state
        {"name": "project_31104", "kind": "project", "tokens": 31104, "k": 4096, "heads": 32,
         "elem": F16},
        # block-sparse attention at the headline size and the default options
        {"name": "vsa_i8_129024", "kind": "vsa", "bits": 8, "t": 32, "h": 42, "w": 96,
         "prefix": 0, "heads": 32, "keep": 10.0, "gate": False},
        # an ordinary ragged grid behind a text prefix, f16 attention, gated
        {"name": "vsa_f16_gated_17704", "kind": "vsa", "bits": 16, "t": 13, "h": 30, "w": 45,
         "prefix": 154, "heads": 32, "keep": 10.0, "gate": True},
        # the INT4 path one past a tile edge
        {"name": "int4_fp6_16385", "kind": "int4", "form": "fp6", "tokens": 16385, "heads": 32,
         "elem": BF16},
    ]


def _log(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]."""
    return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    kind = rng.choice(["short", "short", "fused", "fused", "compact", "cross", "project", "project",
                       "vsa", "vsa", "int4"])
    if kind == "short":
        return {"kind": kind, "tokens": _log(rng, 1, 4095), "heads": 2 * _log(rng, 1, 28),
                "smooth": rng.random() < 0.5, "rope": rng.random() < 0.5}
    if kind == "fused":
        tokens = _log(rng, 4096, 48000)
        return {"kind": kind, "tokens": tokens, "heads": 2 * _log(rng, 2, 28 if tokens < 20000 else 8),
                "elem": rng.choice([F16, BF16]), "smooth": rng.random() < 0.5}
    if kind == "compact":
        tokens = 256 * _log(rng, 17, 64) - rng.randrange(16, 200)
        return {"kind": kind, "tokens": tokens, "heads": 2 * _log(rng, 2, 16),
                "k": 256 * _log(rng, 4, 24)}
    if kind == "cross":
        group = rng.choice([1, 2, 4, 8])
        kv_heads = _log(rng, 1, 32 // group)
        return {"kind": kind, "tokens": _log(rng, 256, 130272), "heads": group * kv_heads,
                "kv_heads": kv_heads, "kv_tokens": _log(rng, 17, 1024),
                "pad": rng.choice([0.0, 0.1, 0.2, 0.5])}
    if kind == "project":
        return {"kind": kind, "tokens": _log(rng, 1, 32000), "k": 256 * _log(rng, 4, 28),
                "heads": 2 * _log(rng, 2, 28), "elem": rng.choice([F16, F32, BF16])}
    if kind == "vsa":
        return {"kind": kind, "bits": rng.choice([8, 16]), "t": _log(rng, 4, 24),
                "h": rng.randrange(16, 41), "w": rng.randrange(24, 65),
                "prefix": rng.choice([0, _log(rng, 32, 1248)]), "heads": 2 * _log(rng, 2, 16),
                "keep": rng.choice([5.0, 10.0, 20.0]), "gate": rng.random() < 0.5}
    return {"kind": kind, "form": rng.choice(["fp6", "ws", "skip"]), "tokens": _log(rng, 1024, 24000),
            "heads": 2 * _log(rng, 2, 16), "elem": rng.choice([F16, BF16])}


# ---------------------------------------------------------------- inputs

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, *shape, dtype=torch.float16):
    return torch.randn(shape, generator=g, device=DEV, dtype=torch.float32).to(dtype)


def _big_randn(g, rows, cols, dtype):
    """N(0, 1), made in pieces so that the f32 copy of a large one stays small."""
    out = torch.empty((rows, cols), dtype=dtype, device=DEV)
    step = max(1, (1 << 27) // cols)
    for r in range(0, rows, step):
        out[r:r + step] = _randn(g, min(step, rows - r), cols, dtype=dtype)
    return out


def _k_offset(g, width, dtype):
    """The per-channel offset keys have in practice, N(0, 2)."""
    return (torch.randn(width, generator=g, device=DEV) * 2.0 ** 0.5).to(dtype)


def _tables(tokens):
    """cos/sin of a (t, h, w) grid walked row by row, 54 cells wide."""
    i = np.arange(tokens, dtype=np.int64)
    pos = np.stack([i // (24 * 54), (i // 54) % 24, i % 54], axis=1).astype(np.float64)
    inv = (10000.0 ** (-np.arange(16) / 16.0)).astype(np.float32)
    cos, sin = H.rope_dit_tables(pos, inv)
    return torch.from_numpy(cos).to(DEV), torch.from_numpy(sin).to(DEV)


def _norms(g):
    w = [torch.rand(128, generator=g, device=DEV) * 0.5 + 0.75 for _ in range(2)]
    return w[0], w[1]


def _qkv(c, g, dtype):
    """The fused projection [tokens][3 * width]."""
    width = c["heads"] * 128
    x = _big_randn(g, c["tokens"], 3 * width, dtype)
    x[:, width:2 * width] += _k_offset(g, width, dtype)
    return x


def _hidden(c, g):
    """A hidden state with a few large channels, as a residual stream has them."""
    x = _big_randn(g, c["tokens"], c["k"], DTYPES[c.get("elem", F16)])
    x[:, :: c["k"] // 8] *= 8
    return x


def _weights(c, g):
    n = 3 * c["heads"] * 128
    w = torch.randint(-127, 128, (n, c["k"]), generator=g, device=DEV, dtype=torch.int8)
    ws = (torch.rand(n, generator=g, device=DEV) * 0.5 + 0.75) * (1.0 / 73.0 / c["k"] ** 0.5)
    return w, ws


def _out(tokens, width):
    return torch.empty((tokens, width), dtype=torch.float16, device=DEV)


def _blocks(c):
    """The plan of the prefix and the grid: H.vsa_plan's arguments."""
    cells = c["t"] * c["h"] * c["w"]
    segments = [(0, c["prefix"])] if c["prefix"] else []
    return segments, c["prefix"] + cells


def prepare(c, seed):
    g = _gen(seed)
    s = {"case": c, "kind": c["kind"]}
    if c["kind"] == "vsa":
        segments, tokens = _blocks(c)
        plan = H.vsa_plan(segments, tokens, c["t"], c["h"], c["w"])
        width = c["heads"] * 128
        s["q"], s["k"], s["v"] = (_big_randn(g, tokens, width, torch.float16) for _ in range(3))
        s["k"] += _k_offset(g, width, torch.float16)
        s["gate"] = _big_randn(g, tokens, width, torch.float16) if c["gate"] else None
        s["out"] = _out(tokens, width)
        s["vsa"] = H.Vsa(*plan, c["heads"], options=H.VsaOptions(keep_percent=c["keep"]),
                         bits=c["bits"])
        return s
    t, heads = c["tokens"], c["heads"]
    width = heads * 128
    s["t"] = t
    if c["kind"] in ("project", "compact"):
        s["x"] = _hidden(c, g)
        s["w"], s["ws"] = _weights(c, g)
        s["plain"] = H.PreparePlainCfg(c["k"], 256, c["k"], ELEMS[c.get("elem", F16)])
        s["gemm"] = H.GemmCfg(c["k"], 3 * width, c["k"], 4)
        s["codes"] = torch.empty((t, c["k"]), dtype=torch.int8, device=DEV)
        s["scales"] = torch.empty(t, dtype=torch.float32, device=DEV)
        s["qkv"] = torch.empty(H.compact_qkv_elements(t, 3 * width), dtype=torch.float16, device=DEV)
    if c["kind"] in ("fused", "compact"):
        elem = c.get("elem", F16)
        if c["kind"] == "fused":
            s["qkv"] = _qkv(c, g, DTYPES[elem])
        s["qn"], s["kn"] = _norms(g)
        s["cos"], s["sin"] = _tables(t)
        s["out"] = _out(t, width)
        s["stack"] = H.Stack(heads, t, eps=EPS, elem=ELEMS[elem], ksmooth=c.get("smooth", False))
    elif c["kind"] == "short":
        if c["rope"]:
            s["qkv"] = _qkv(c, g, torch.float16)
            s["qn"], s["kn"] = _norms(g)
            s["cos"], s["sin"] = _tables(t)
            s["rope"] = H.RopeCfg(3 * width, heads, heads, width, EPS, 1, H.H3_ELEM_F16)
            s["q"], s["k"], s["v"] = (_out(t, width) for _ in range(3))
        else:
            x = _qkv(c, g, torch.float16)
            s["q"], s["k"], s["v"] = (x[:, i * width:(i + 1) * width].contiguous() for i in range(3))
        s["out"] = _out(t, width)
        s["stack"] = H.Stack(heads, t, eps=EPS, ksmooth=c["smooth"], fused=False)
    elif c["kind"] == "cross":
        kh, kt = c["kv_heads"], c["kv_tokens"]
        kcap, cap = -(-kt // 32) * 32, -(-t // 32) * 32
        s["q"] = _big_randn(g, t, width, torch.float16)
        s["k"], s["v"] = _randn(g, kt, kh * 128), _randn(g, kt, kh * 128)
        s["mask"] = (torch.arange(kt, device=DEV) < max(1, int(kt * (1 - c["pad"])))).to(torch.uint8)
        s["ki"] = torch.zeros(kh * kcap * 32, dtype=torch.int32, device=DEV)
        s["ks"] = torch.zeros(kh * kcap, dtype=torch.float32, device=DEV)
        s["vt"] = torch.zeros(kh * 128 * kcap, dtype=torch.float16, device=DEV)
        # the text's operands: once per prompt
        H.prepare_qk_i8hm(H.PrepareCfg(kh * 128, 0, kh, 1.0, kcap, EPS, H.H3_ELEM_F16), kt, s["k"],
                          None, s["ki"], s["ks"])
        H.transpose_f16(H.TransposeCfg(kh * 128, kcap, H.H3_ELEM_F16), kcap, kt, s["v"], s["vt"])
        s["qi"] = torch.zeros(heads * cap * 32, dtype=torch.int32, device=DEV)
        s["qs"] = torch.zeros(heads * cap, dtype=torch.float32, device=DEV)
        s["prep"] = H.PrepareCfg(width, 0, heads, H.EXTRA_Q, cap, EPS, H.H3_ELEM_F16)
        s["cfg"] = H.CrossCfg(heads, kh, t, cap, kt, kcap, width)
        s["out"] = _out(t, width)
    elif c["kind"] == "int4":
        cap = H.capacity(t)
        s["qkv"] = _qkv(c, g, DTYPES[c["elem"]])
        s["qi"], s["ki"] = (torch.zeros((cap, width // 8), dtype=torch.int32, device=DEV)
                            for _ in range(2))
        s["qs"], s["ks"] = (torch.zeros((cap, heads), dtype=torch.float32, device=DEV)
                            for _ in range(2))
        s["vt"] = torch.zeros((width, cap), dtype=torch.float16, device=DEV)
        s["pq"] = H.PrepareCfg(3 * width, 0, heads, H.EXTRA_Q, cap, EPS, ELEMS[c["elem"]])
        s["pk"] = H.PrepareCfg(3 * width, width, heads, 1.0, cap, EPS, ELEMS[c["elem"]])
        s["tr"] = H.TransposeCfg(width, cap, ELEMS[c["elem"]])
        if c["form"] == "skip":
            s["cfg"] = H.AttentionSkipCfg(width, width, width, t, cap, 1.0, SKIP_TAU)
        else:
            s["cfg"] = H.AttentionCfg(width, width, width, t, cap, 1.0)
        size = (H.fp6_workspace_bytes if c["form"] == "fp6" else H.scales_workspace_bytes)(s["cfg"])
        s["lent"] = torch.empty(size, dtype=torch.uint8, device=DEV)
        s["out"] = _out(t, width)
    return s


SKIP_TAU = 40.0  # natural-log units: a skipped tile holds less than e^-40 of a row


# ---------------------------------------------------------------- one pass

def run(s):
    kind = s["kind"]
    if kind == "vsa":
        s["vsa"].attend(0, s["q"], s["k"], s["v"], s["out"], s["gate"])
        return s["out"]
    t = s["t"]
    if kind == "short":
        if "rope" in s:
            H.rope_qknorm_f16(s["rope"], t, s["qkv"], s["qn"], s["kn"], s["cos"], s["sin"], s["q"],
                              s["k"], s["v"])
        s["stack"].attend(t, s["q"], s["k"], s["v"], s["out"])
        return s["out"]
    if kind == "fused":
        s["stack"].attend_fused(t, s["qkv"], s["qn"], s["kn"], s["cos"], s["sin"], s["out"])
        return s["out"]
    if kind == "cross":
        H.prepare_qk_i8hm(s["prep"], t, s["q"], None, s["qi"], s["qs"])
        H.attention_i8qkhm_cross(s["cfg"], s["qi"], s["qs"], s["ki"], s["ks"], s["vt"], s["mask"],
                                 s["out"])
        return s["out"]
    if kind == "int4":
        H.prepare_qk_i4(s["pq"], t, s["qkv"], None, s["qi"], s["qs"])
        H.prepare_qk_i4(s["pk"], t, s["qkv"], None, s["ki"], s["ks"])
        H.transpose_qkv_v_f16(s["tr"], s["tr"].row_capacity, t, s["qkv"], s["vt"])
        attend = {"fp6": H.attention_i4qk_fp6, "ws": H.attention_i4qk_ws,
                  "skip": H.attention_i4qks_ws}[s["case"]["form"]]
        attend(s["cfg"], t, s["case"]["heads"], s["qi"], s["qs"], s["ki"], s["ks"], s["vt"],
               s["out"], s["lent"])
        return s["out"]
    H.prepare_plain_i8(s["plain"], t, s["x"], s["codes"], s["scales"])
    H.gemm_i8_qkv_256(s["gemm"], t, s["codes"], s["w"], s["ws"], s["scales"], s["qkv"])
    if kind == "project":
        return s["qkv"]
    s["stack"].attend_compact(t, s["qkv"], s["qn"], s["kn"], s["cos"], s["sin"], s["out"])
    return s["out"]


# ---------------------------------------------------------------- what a pass cannot do without

def _kept_share(c):
    """The share of the (query block, key block) pairs the default routing keeps, and blocks."""
    prefix = -(-c["prefix"] // 64)
    cubes = -(-c["t"] // 4) * -(-c["h"] // 4) * -(-c["w"] // 4)
    n = prefix + cubes
    kept = prefix * n + cubes * min(n, prefix + max(1, min(cubes - 1, round(c["keep"] / 100 * cubes))) + 2)
    return kept / (n * n)


def work(c):
    heads = c["heads"]
    width = heads * 128
    if c["kind"] == "vsa":
        tokens = _blocks(c)[1]
        io = tokens * width * 2 * (5 if c["gate"] else 4)
        return {"bytes": io, "flops": 4.0 * tokens * tokens * width * _kept_share(c)}
    t = c["tokens"]
    attention = 4.0 * t * t * width
    if c["kind"] == "cross":
        return {"bytes": t * width * 4 + c["kv_heads"] * c["kv_tokens"] * 388,
                "flops": 4.0 * t * c["kv_tokens"] * width}
    if c["kind"] in ("project", "compact"):
        x = t * c["k"] * (4 if c.get("elem") == F32 else 2) + 3 * width * c["k"]
        gemm = 2.0 * t * 3 * width * c["k"]
        if c["kind"] == "project":
            return {"bytes": x + t * 3 * width * 2, "flops": gemm}
        return {"bytes": x + t * (width * 2 + 384), "flops": gemm + attention}
    # q, k, v read and the output written, and RoPE's tables
    return {"bytes": t * width * 8 + (t * 384 if c["kind"] == "fused" or c.get("rope") else 0),
            "flops": attention}


def tolerance(c):
    if c["kind"] == "project":
        return "exact"  # integer codes and sums, and an epilogue of named f32 operations
    # f16 probabilities against f16 values and an f16 result: 2.9e-4 to 4.0e-4 from the same in 64
    # bits over these ranges (where a rounding tie moves a code or a route, as the 64-bit form's
    # quantizer and means do now and then, 1e-3 to 2e-3: such moves are not the attention's).
    return {"rel": 1.5e-3}


# ---------------------------------------------------------------- the same in 64 bits

def _sylvester(n):
    h = torch.ones((1, 1), dtype=torch.float64, device=DEV)
    while h.shape[0] < n:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return h


def _quantized(x, extra=1.0, top=127):
    """[tokens][128] rows rotated and quantized, as the values their codes stand for."""
    r = x @ _sylvester(128)
    amax = r.abs().amax(1, keepdim=True).clamp_min(1e-30)
    return torch.round(r * (top / amax)).clamp(-top, top) * (amax / top * extra)


def _softmax_av(q, k, v, mask_of=None):
    """softmax(q k^T) v of one head in pieces of rows; mask_of(r0, r1): the keys each row sees."""
    out = torch.empty((q.shape[0], v.shape[1]), dtype=torch.float64, device=DEV)
    step = max(1, (1 << 27) // k.shape[0])
    for r in range(0, q.shape[0], step):
        s = q[r:r + step] @ k.t()
        if mask_of is not None:
            s.masked_fill_(~mask_of(r, min(r + step, q.shape[0])), -float("inf"))
        out[r:r + step] = torch.softmax(s, 1) @ v
    return out


def _roped(x, w, cos, sin):
    """RMSNorm and rotate-half RoPE of [tokens][128] rows, rounded to f16."""
    x = x * torch.rsqrt(x.square().mean(1, keepdim=True) + EPS) * w.double()
    a, b, cos, sin = x[:, :48], x[:, 48:96], cos.double(), sin.double()
    return torch.cat([a * cos - b * sin, b * cos + a * sin, x[:, 96:]], 1).half().double()


def _group_hadamard():
    h4 = torch.tensor([[1, 1, 1, -1], [1, 1, -1, 1], [1, -1, 1, 1], [-1, 1, 1, 1]],
                      dtype=torch.float64, device=DEV)
    h = h4
    for _ in range(3):
        h = torch.kron(h, h4)
    return h


def _projected(c, s):
    """(Q and K rows [tokens][2 width], V [tokens][width]) of the projection, f16 values."""
    x = s["x"].double().view(c["tokens"], -1, 256) @ _group_hadamard()
    x = x.view(c["tokens"], -1) / 16
    sc = x.abs().amax(1, keepdim=True).clamp_min(1e-30) / 127
    a = torch.round(x / sc).clamp(-127, 127)
    out = torch.empty((c["tokens"], s["w"].shape[0]), dtype=torch.float16, device=DEV)
    for n in range(0, s["w"].shape[0], 4096):
        y = (a @ s["w"][n:n + 4096].double().t()) * s["ws"][n:n + 4096].double() * sc
        out[:, n:n + 4096] = y.half()
    two = s["w"].shape[0] // 3 * 2
    return out[:, :two].contiguous(), out[:, two:].contiguous()


def _block_of(c):
    """The block of each token, the blocks, and how many of them hold the prefix."""
    p = c["prefix"]
    prefix = -(-p // 64)
    i = torch.arange(c["t"] * c["h"] * c["w"], device=DEV)
    t, h, w = i // (c["h"] * c["w"]) // 4, i // c["w"] % c["h"] // 4, i % c["w"] // 4
    nh, nw = -(-c["h"] // 4), -(-c["w"] // 4)
    cube = prefix + (t * nh + h) * nw + w
    return torch.cat([torch.arange(p, device=DEV) // 64, cube]), prefix + -(-c["t"] // 4) * nh * nw, prefix


def _exact_vsa(c, s):
    of, n, prefix = _block_of(c)
    cubes = n - prefix
    topk = max(1, min(cubes - 1, round(c["keep"] / 100 * cubes)))
    live = torch.bincount(of, minlength=n).double()[:, None]
    near = torch.arange(n, device=DEV)
    forced = (near[:, None] - near[None]).abs() <= 1
    forced[:prefix] = True
    forced[:, :prefix] = True
    out = torch.empty((len(of), c["heads"] * 128), dtype=torch.float64, device=DEV)
    for h in range(c["heads"]):
        q, k, v = (s[x][:, 128 * h:128 * h + 128].double() for x in "qkv")
        qm, km, vm = (torch.zeros((n, 128), dtype=torch.float64, device=DEV).index_add_(0, of, x) / live
                      for x in (q, k, v))
        scores = qm @ km.t()
        least = scores[:, prefix:].topk(topk, 1).values[:, -1:]
        kept = forced | (scores >= least)
        if c["bits"] == 8:
            q, k = _quantized(q, 128 ** -0.5 / 128), _quantized(k)
        else:
            q = q * 128 ** -0.5
        y = _softmax_av(q, k, v, lambda a, b: kept[of[a:b]][:, of])
        if c["gate"]:
            coarse = torch.softmax(scores * 128 ** -0.5, 1) @ vm
            y += s["gate"][:, 128 * h:128 * h + 128].double() * coarse[of]
        out[:, 128 * h:128 * h + 128] = y
    return out


def exact(c, seed):
    tokens = _blocks(c)[1] if c["kind"] == "vsa" else c["tokens"]
    keys = c["kv_tokens"] if c["kind"] == "cross" else tokens
    if c["kind"] != "project" and float(tokens) * keys * c["heads"] > 6e10:
        return None
    s = prepare(c, seed)
    if c["kind"] == "vsa":
        return _exact_vsa(c, s)
    heads = c["heads"]
    width = heads * 128
    if c["kind"] in ("project", "compact"):
        qk, v = _projected(c, s)
        if c["kind"] == "project":
            cap = -(-tokens // 256) * 256
            vt = torch.zeros((width, cap), dtype=torch.float16, device=DEV)
            vt[:, :tokens] = v.t()
            return torch.cat([qk.reshape(-1), vt.reshape(-1)]).double()
        qkv = torch.cat([qk, v], 1)
    elif c["kind"] == "cross":
        qkv = None
    else:
        qkv = s["qkv"] if "qkv" in s else torch.cat([s["q"], s["k"], s["v"]], 1)
    extra = 128 ** -0.5 / 128
    out = torch.empty((tokens, width), dtype=torch.float64, device=DEV)
    for h in range(heads):
        if c["kind"] == "cross":
            kh = h // (heads // c["kv_heads"])
            q = s["q"][:, 128 * h:128 * h + 128].double()
            k, v = (s[x][:, 128 * kh:128 * kh + 128].double() for x in "kv")
        else:
            q, k, v = (qkv[:, i * width + 128 * h:i * width + 128 * h + 128].double() for i in range(3))
            v = v.half().double()
        if "cos" in s:
            q, k = _roped(q, s["qn"], s["cos"], s["sin"]), _roped(k, s["kn"], s["cos"], s["sin"])
        if c.get("smooth"):
            k = k - k.mean(0, keepdim=True)
        top = 7 if c["kind"] == "int4" else 127
        q, k = _quantized(q, extra, top), _quantized(k, 1.0, top)
        mask_of = (lambda a, b: (s["mask"] != 0)[None]) if c["kind"] == "cross" else None
        out[:, 128 * h:128 * h + 128] = _softmax_av(q, k, v, mask_of)
    return out
