"""Attention calls whose query blocks do not fill the chip, or leave a partial last round, run (in
part) on the key-split kernel: the ways a call is divided, at the edges of its tiles and units,
against the f64 oracle at the head-major suite's bar (1e-3 + 2e-3 rel), in every operand layout the
dispatch accepts. Both layouts divide a call alike and the kernel reads them through pitches, so
their outputs agree bit for bit."""
import numpy as np
import pytest

import h3attn as H
import oracle as O
from helpers import filled, head_major_operands, pack_codes, to_dev

pytestmark = pytest.mark.gpu


# (tokens, token_count, query heads, key/value heads, pad): fewer stages than key groups; one row,
# one key past a stage, a wave with no live row; every number of tiles in a last block; a chip-filling
# count of full blocks with a partial one left over; head wrap and padded output pitches
@pytest.mark.parametrize("tokens,count,q_heads,kv_heads,pad", [
    (1, 1, 2, 2, 0), (33, 33, 3, 3, 128), (65, 65, 2, 2, 0), (129, 129, 56, 56, 0),
    (257, 256, 8, 8, 0), (512, 449, 4, 2, 128), (1000, 1000, 7, 7, 0), (1024, 1024, 8, 8, 128),
    (2047, 2047, 8, 8, 0), (4160, 300, 5, 5, 0), (8193, 8193, 16, 16, 0)])
def test_divided_calls_match_the_oracle_in_both_layouts(dev, tokens, count, q_heads, kv_heads, pad):
    import torch

    cap = O.capacity(tokens)
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
