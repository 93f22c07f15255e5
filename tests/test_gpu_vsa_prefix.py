"""The VSA runtime's prefix cubes run apart from the video cubes where that is faster, each split into
ranges of the key cubes whose partial results are combined, or whole where there are many. On the
runtime's own operands and routes its gathered output is held against the public attention entry, which
knows no prefix and walks every query cube in one piece: the video cubes' rows, and rows of cubes that are
not split, are the same bits, the split cubes' rows agree to a few f16 roundings."""
import numpy as np
import pytest

import h3attn as H
from helpers import read_device, vsa_prefix

pytestmark = pytest.mark.gpu


# plans whose prefix is no longer than other cubes' lists for its share of the call, in one order (0, 1):
# one partial cube, many cubes, few key cubes, nearly all prefix; and apart: one partial cube, three cubes
# with a partial one, ranges of fewer than nine key cubes, eleven cubes, more cubes than one generation
# of workgroups takes (whole), and a plan whose video cubes, more than three generations, are one launch
@pytest.mark.parametrize("bits", [8, 16])
@pytest.mark.parametrize("segments,grid,heads,apart", [
    ([(0, 5)], (8, 12, 13), 2, (0, 1)), ([(0, 2112)], (4, 16, 16), 32, (0, 1)),
    ([(0, 64)], (4, 8, 4), 2, (0, 1)), ([(0, 700)], (4, 5, 4), 2, (0, 1)),
    ([(0, 5)], (12, 20, 24), 2, (1, 11)), ([(0, 77), (77, 70)], (9, 16, 17), 3, (4, 8)),
    ([(0, 64)], (8, 20, 20), 2, (1, 6)), ([(0, 700)], (8, 24, 32), 2, (11, 13)),
    ([(0, 2112)], (12, 32, 32), 32, (33, 1)), ([(0, 30)], (9, 25, 26), 24, (1, 16))])
def test_runtime_prefix_cubes_match_the_whole_walk(dev, bits, segments, grid, heads, apart):
    import torch

    rows = sum(n for _, n in segments) + int(np.prod(grid))
    width = heads * 128
    src, inverse, lengths, prefix = H.vsa_plan(segments, rows, *grid)
    assert vsa_prefix(heads, prefix, len(lengths),
                      H.VsaOptions().topk(len(lengths) - prefix)) == apart
    vsa = H.Vsa(src, inverse, lengths, prefix, heads, bits=bits)
    g = torch.Generator(device=dev).manual_seed(rows + bits)
    q, k, v = (torch.randn((rows, width), generator=g, device=dev).half() for _ in range(3))
    out = torch.empty((rows, width), dtype=torch.float16, device=dev)
    print(f"prefix cubes: bits={bits} segments={segments} grid={grid} heads={heads}", flush=True)
    vsa.attend(0, q, k, v, out)
    b = vsa.buffers(0)
    padded = b.cfg.padded
    whole = torch.empty((padded, width), dtype=torch.float16, device=dev)
    if bits == 8:
        H.vsa_attention_i8(b.attention, padded, heads, b.qi, b.qs, b.ki, b.ks, b.vt, whole, b.routes,
                           b.lengths)
    else:
        H.vsa_attention_f16(b.attention, padded, heads, b.q, b.k, b.v, whole, b.routes, b.lengths)
    torch.cuda.synchronize()
    got = read_device(b.out).view(np.float16).reshape(padded, width)
    want = whole.cpu().numpy()
    live = (np.arange(64)[None] < lengths[:, None]).reshape(-1)  # dead rows hold no result to compare
    exact = 64 * prefix if apart[1] > 1 else 0  # first row of cubes that were walked in one piece
    assert np.array_equal(got[exact:][live[exact:]].view(np.uint16),
                          want[exact:][live[exact:]].view(np.uint16))
    a, w = (x[:64 * prefix][live[:64 * prefix]].astype(np.float64) for x in (got, want))
    # both forms: f16 probabilities (2^-11) against |v| <= 4.5, pair sums in f16 (2^-9) and an f16 result
    assert np.isfinite(a).all()
    assert np.all(np.abs(a - w) <= 2.0 ** -10 * np.abs(w) + 4.5 * 2.0 ** -9), float(np.abs(a - w).max())
    again = torch.empty_like(out)
    vsa.reset()
    vsa.attend(0, q, k, v, again)
    torch.cuda.synchronize()
    assert torch.equal(out, again)
