"""Attention calls whose query blocks do not fill the chip, or leave a partial last round, run (in
part) on the key-split kernel: the ways a call is divided, at the edges of its tiles and units,
against the f64 oracle at the head-major suite's bar (1e-3 + 2e-3 rel) in both INT8 layouts, and in the
FP6 form at its suite's. Both layouts divide a call alike and the kernel reads them through pitches, so
their outputs agree bit for bit. Every case asserts how the rule divides it."""
import numpy as np
import pytest

import h3attn as H
import oracle as O
from helpers import (filled, from_dev, head_major_operands, north_star_ok, pack_codes, split_plan,
                     to_dev)
from test_gpu_fp6 import operands, oracle_rows, run_fp6
from test_gpu_i4 import pack_i4

pytestmark = pytest.mark.gpu


# (tokens, token_count, query heads, key/value heads, pad) and the division, None for undivided or (blocks on
# the undivided kernel, tiles per unit of the other full blocks, of the last, partial blocks): calls of one
# stage, and of three whose units would be more than the chip holds; two, three and seven stages (idle key
# groups); one key past eight stages; one to eight live tiles in the last block; only whole blocks; a wave
# with no live row; units of two tiles; whole rounds with the partial blocks, with a round of full blocks, and
# with both left over; head wrap and padded output pitches
CASES = [
    (1, 1, 2, 2, 0, None), (33, 33, 3, 3, 128, None), (129, 129, 56, 56, 0, None),
    (65, 65, 2, 2, 0, (0, 1, 1)), (129, 129, 5, 5, 128, (0, 1, 1)), (257, 256, 8, 8, 0, (0, 1, 1)),
    (385, 385, 2, 2, 0, (0, 1, 1)), (447, 447, 3, 3, 0, (0, 1, 1)), (448, 448, 5, 5, 0, (0, 1, 1)),
    (449, 449, 3, 3, 0, (0, 1, 1)), (512, 449, 4, 2, 128, (0, 1, 1)), (513, 513, 4, 4, 0, (0, 1, 1)),
    (577, 545, 4, 4, 0, (0, 1, 1)), (640, 609, 2, 2, 128, (0, 1, 1)), (200, 161, 4, 4, 0, (0, 1, 1)),
    (1000, 1000, 7, 7, 0, (0, 1, 1)), (1024, 1024, 8, 8, 128, (0, 1, 1)),
    (2047, 2047, 8, 8, 0, None), (4160, 300, 5, 5, 0, (0, 1, 1)), (2816, 2816, 3, 3, 0, (0, 2, 1)),
    (2806, 2806, 3, 3, 0, (0, 2, 2)), (4858, 184, 50, 50, 0, (0, 1, 2)),
    (4864, 4864, 14, 14, 0, (256, 1, 1)), (8193, 8193, 16, 16, 0, (512, 1, 1)),
    (34007, 34007, 2, 2, 0, (256, 1, 1))]


def check_division(tokens, count, heads, plan, cap=None):
    got = split_plan(tokens, count, heads, cap or H.capacity(tokens))
    assert got == plan, got


@pytest.mark.parametrize("tokens,count,q_heads,kv_heads,pad,plan", CASES)
def test_divided_calls_match_the_oracle_in_both_layouts(dev, tokens, count, q_heads, kv_heads, pad,
                                                        plan):
    check_against_the_oracle(dev, tokens, count, q_heads, kv_heads, pad, plan, O.capacity(tokens))


# capacities are multiples of 16, so V^T's rows begin at any 32 bytes of a 128-byte line: 96 (1,008 and 1,072),
# 32 and, with no room for another token, 64
@pytest.mark.parametrize("tokens,count,q_heads,kv_heads,cap", [
    (1000, 1000, 7, 7, 1008), (1000, 999, 4, 2, 1040), (480, 480, 5, 5, 480), (1025, 1025, 3, 3, 1072)])
def test_divided_calls_at_any_capacity(dev, tokens, count, q_heads, kv_heads, cap):
    check_against_the_oracle(dev, tokens, count, q_heads, kv_heads, 0, (0, 1, 1), cap)


def check_against_the_oracle(dev, tokens, count, q_heads, kv_heads, pad, plan, cap):
    import torch

    check_division(tokens, count, q_heads, plan, cap)
    rng = np.random.default_rng(tokens + 13 * q_heads)
    qc, qs, _, _, _ = head_major_operands(rng, q_heads, tokens, cap, late_match=False)
    _, _, kc, ks, vt = head_major_operands(rng, kv_heads, tokens, cap, late_match=False)
    kc[:, tokens - 1] = qc[:kv_heads, min(31, tokens - 1)]  # a strong match in the last key
    out_stride = q_heads * 128 + pad
    cfg = H.AttentionCfg(q_heads * 128, kv_heads * 128, out_stride, tokens, cap, 1.0)
    hm = [to_dev(pack_codes(qc).reshape(q_heads * cap, 32), dev), to_dev(qs, dev),
          to_dev(pack_codes(kc).reshape(kv_heads * cap, 32), dev), to_dev(ks, dev)]
    tm = [to_dev(pack_codes(qc.transpose(1, 0, 2)).reshape(cap, q_heads * 32), dev),
          to_dev(qs.T.copy(), dev),
          to_dev(pack_codes(kc.transpose(1, 0, 2)).reshape(cap, kv_heads * 32), dev),
          to_dev(ks.T.copy(), dev)]
    vt_d = to_dev(vt, dev)
    ws = torch.empty(H.scales_workspace_bytes(cfg), dtype=torch.uint8, device=dev)
    nbytes = count * out_stride * 2
    print(f"divided call: S={tokens} rows={count} heads={q_heads}/{kv_heads} pad={pad}", flush=True)

    def run(fn, ops, *lent):
        out = filled((nbytes + 64,), 0xA5, np.uint8, dev)  # a guard past the last row
        fn(cfg, count, q_heads, *ops, vt_d, out[:nbytes], *lent)
        torch.cuda.synchronize()
        host = out.cpu().numpy()
        assert (host[nbytes:] == 0xA5).all(), "written past the output"
        return host[:nbytes]

    got = run(H.attention_i8qkhm, hm)
    for fn, ops, lent in ((H.attention_i8qkhm, hm, ()), (H.attention_i8qk, tm, ()),
                          (H.attention_i8qk_ws, tm, (ws,))):
        assert np.array_equal(got, run(fn, ops, *lent)), fn.__name__
    touched = min(kv_heads, out_stride // 128)
    rows_out = got.view(np.uint16).reshape(count, out_stride)
    assert (rows_out[:, touched * 128:] == 0xA5A5).all(), "untouched heads or pad columns written"
    values = rows_out[:, :touched * 128].view(np.float16).astype(np.float64)
    assert np.isfinite(values).all()
    rows = np.unique(np.concatenate([[0, min(31, count - 1), (count - 1) // 32 * 32, count - 1],
                                     rng.integers(0, count, 5)])).astype(np.int32)
    want = O.attention_f64(qc[:touched], qs[:touched], kc[:touched], ks[:touched],
                           vt[:touched * 128], tokens, cap, touched, rows)
    err = np.abs(values.reshape(count, touched, 128)[rows] - want)
    assert np.all(err <= 1e-3 + 2e-3 * np.abs(want)), float(err.max())


@pytest.mark.parametrize("tokens,count,heads,plan", [
    (c[0], c[1], c[2], c[5]) for c in CASES if c[2] == c[3] and c[4] == 0 and c[5] and c[0] < 10000])
def test_divided_fp6_calls_match_the_oracle(dev, tokens, count, heads, plan):
    import torch

    check_division(tokens, count, heads, plan)
    cap = H.capacity(tokens)
    rng = np.random.default_rng(tokens + 31 * heads)
    q, k, qs, ks, vt = operands(rng, tokens, heads, cap)
    print(f"divided FP6 call: S={tokens} rows={count} heads={heads}", flush=True)
    got, _, cfg = run_fp6(dev, q, qs, k, ks, vt, tokens, cap, heads, token_count=count)
    a6 = got.view(np.float16).astype(np.float64)
    assert np.isfinite(a6).all()
    rows = np.unique(np.concatenate([[0, min(31, count - 1), count - 1],
                                     rng.integers(0, count, 5)])).astype(np.int32)
    want = oracle_rows(q, qs, k, ks, vt, tokens, cap, heads, rows)
    mx, mean = north_star_ok(a6.reshape(count, heads, 128)[rows], want)
    assert mx <= 2e-2 and mean <= 2e-3, (mx, mean)
    # every row against the int8-MFMA int4 kernel, which divides no call
    out4 = torch.zeros((count, heads * 128), dtype=torch.float16, device=dev)
    H.attention_i4qk(cfg, count, heads, to_dev(pack_i4(q), dev), to_dev(qs, dev),
                     to_dev(pack_i4(k), dev), to_dev(ks, dev), to_dev(vt, dev), out4)
    a4 = from_dev(out4).view(np.float16).astype(np.float64)
    assert np.all(np.abs(a6 - a4) <= 2e-3 + 4e-3 * np.abs(a4))
