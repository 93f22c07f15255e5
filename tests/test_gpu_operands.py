"""The Stack's operands come from one launch per call: held bit for bit against the public entries it
stands for (two quantizers and a transpose), at the edges of its workgroups (rows in flight, chunks of
heads, 64-column tiles), and the column mean's two kernels against the oracle at their boundary."""
import numpy as np
import pytest

import h3attn as H
import oracle as O
from helpers import from_dev, read_device, to_dev

pytestmark = pytest.mark.gpu


def bindings(stack):
    ops = stack.operands()
    return {n: read_device(getattr(ops, n)) for n in ("qi", "ki", "qs", "ks", "vt")}


# token-major with one row and with four rows in flight per group, and head-major
@pytest.mark.parametrize("smooth", [False, True])
@pytest.mark.parametrize("tokens,heads,bf16", [(1, 2, False), (33, 4, True), (129, 56, False),
                                               (585, 56, True), (4097, 6, False)])
def test_separate_operands_match_the_public_entries(dev, tokens, heads, bf16, smooth):
    import torch

    width, elem = heads * 128, H.H3_ELEM_BF16 if bf16 else H.H3_ELEM_F16
    dtype = torch.bfloat16 if bf16 else torch.float16
    g = torch.Generator(device=dev).manual_seed(tokens + heads)
    q, k, v = (torch.randn((tokens, width), generator=g, device=dev).to(dtype) for _ in range(3))
    out = torch.empty((tokens, width), dtype=torch.float16, device=dev)
    stack = H.Stack(heads, tokens, elem=elem, ksmooth=smooth, fused=False)
    print(f"separate operands: {tokens} x {heads} bf16={bf16} smooth={smooth}", flush=True)
    stack.attend(tokens, q, k, v, out)
    got = bindings(stack)
    cap, hm = stack.capacity, bool(stack.operands().head_major)
    zero = torch.zeros(width, device=dev)
    mean = zero
    if smooth:
        mean = torch.empty(width, device=dev)
        H.colmean_f32(width, tokens, k, mean, elem)
    prep = H.prepare_qk_i8hm if hm else H.prepare_qk_i8
    for x, m, extra, codes, scales in ((q, zero, H.EXTRA_Q, "qi", "qs"), (k, mean, 1.0, "ki", "ks")):
        c = torch.zeros(cap * width // 4, dtype=torch.int32, device=dev)
        s = torch.zeros(cap * heads, dtype=torch.float32, device=dev)
        prep(H.PrepareCfg(width, 0, heads, extra, cap if hm else 0, 1e-5, elem), tokens, x, m, c, s)
        assert np.array_equal(got[codes], from_dev(c).view(np.uint8)), codes
        assert np.array_equal(got[scales], from_dev(s).view(np.uint8)), scales
    vt = torch.zeros(width * cap, dtype=torch.float16, device=dev)
    H.transpose_f16(H.TransposeCfg(width, cap, elem), cap, tokens, v, vt)
    assert np.array_equal(got["vt"], from_dev(vt).view(np.uint8)), "vt"


# chunks of 4 heads (a last one of 1), of 8 (a last one of 3), and whole walks
@pytest.mark.parametrize("tokens,heads,bf16", [(4097, 5, False), (5000, 51, True), (65537, 3, False)])
def test_fused_operands_match_the_public_entries(dev, tokens, heads, bf16):
    import torch

    width, elem = heads * 128, H.H3_ELEM_BF16 if bf16 else H.H3_ELEM_F16
    g = torch.Generator(device=dev).manual_seed(tokens + heads)
    x = torch.randn((tokens, 3 * width), generator=g, device=dev).to(
        torch.bfloat16 if bf16 else torch.float16)
    qn, kn = (torch.rand(128, generator=g, device=dev) + 0.5 for _ in range(2))
    ang = torch.rand((tokens, 48), generator=g, device=dev) * 6
    cos, sin = torch.cos(ang), torch.sin(ang)
    out = torch.empty((tokens, width), dtype=torch.float16, device=dev)
    stack = H.Stack(heads, tokens, elem=elem)
    print(f"fused operands: {tokens} x {heads} bf16={bf16}", flush=True)
    stack.attend_fused(tokens, x, qn, kn, cos, sin, out)
    got = bindings(stack)
    cap = stack.capacity
    # the public quantizer, one head at a time: no chunk of heads in it
    for first, w, extra, codes, scales in ((0, qn, H.EXTRA_Q, "qi", "qs"),
                                           (width, kn, 1.0, "ki", "ks")):
        for h in range(heads):
            c = torch.zeros(cap * 32, dtype=torch.int32, device=dev)
            s = torch.zeros(cap, dtype=torch.float32, device=dev)
            H.prepare_qk_rope_i8hm(H.PrepareCfg(3 * width, first + 128 * h, 1, extra, cap, 1e-5, elem),
                                   tokens, x, w, cos, sin, c, s)
            assert np.array_equal(got[codes][cap * 128 * h:cap * 128 * (h + 1)],
                                  from_dev(c).view(np.uint8)), (codes, h)
            assert np.array_equal(got[scales][cap * 4 * h:cap * 4 * (h + 1)],
                                  from_dev(s).view(np.uint8)), (scales, h)
    vt = torch.zeros(width * cap, dtype=torch.float16, device=dev)
    H.transpose_qkv_v_f16(H.TransposeCfg(width, cap, elem), tokens, tokens, x, vt)
    assert np.array_equal(got["vt"], from_dev(vt).view(np.uint8)), "vt"


# the plain kernel's last length and the chain kernel's first; whole, one-over and partial chunks of
# 384 tokens; an input that is 2-byte aligned only
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("tokens,width,bf16", [(192, 256, False), (193, 256, True), (384, 512, False),
                                               (385, 256, False), (1183, 768, True)])
def test_colmean_kernels_are_bit_exact(dev, tokens, width, bf16, offset):
    import torch

    rng = np.random.default_rng(tokens + width)
    f = (rng.standard_normal((tokens, width)) * 3).astype(np.float32)
    bits = (f.view(np.uint32) >> 16).astype(np.uint16) if bf16 else O.f16_bits(f)
    flat = torch.zeros(tokens * width + offset, dtype=torch.int16, device=dev)
    flat[offset:] = to_dev(bits.reshape(-1), dev)
    mean = torch.empty(width, dtype=torch.float32, device=dev)
    print(f"colmean {tokens} x {width} bf16={bf16} offset={offset}", flush=True)
    H.colmean_f32(width, tokens, flat[offset:], mean, H.H3_ELEM_BF16 if bf16 else H.H3_ELEM_F16)
    want = O.colmean(bits, O.BF16 if bf16 else O.F16, tokens, width, width)
    assert np.array_equal(from_dev(mean).view(np.uint32), want.view(np.uint32))
