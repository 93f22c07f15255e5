"""The VSA runtime's prefix cubes run apart from the video cubes, each split into ranges of the key
cubes whose partial results are combined, or whole where there are many. On the runtime's own operands
and routes its gathered output is held against the public attention entry, which knows no prefix and
walks every query cube in one piece: the video cubes' rows are the same bits, the prefix cubes' rows
agree to a few f16 roundings."""
import numpy as np
import pytest

import h3attn as H
from helpers import read_device

pytestmark = pytest.mark.gpu


# prefix rows of one partial cube, of three cubes with a partial one (splits), of more cubes than one
# generation of workgroups takes (no split), a plan of few key cubes (fewer than eight to a range), a
# plan that is nearly all prefix, and one whose video cubes, more than three generations of them, are
# one launch of the runtime
@pytest.mark.parametrize("bits", [8, 16])
@pytest.mark.parametrize("segments,grid,heads", [
    ([(0, 5)], (8, 12, 13), 2), ([(0, 77), (77, 70)], (9, 16, 17), 3), ([(0, 2112)], (4, 16, 16), 32),
    ([(0, 64)], (4, 8, 4), 2), ([(0, 700)], (4, 5, 4), 2), ([(0, 30)], (9, 25, 26), 24)])
def test_runtime_prefix_cubes_match_the_whole_walk(dev, bits, segments, grid, heads):
    import torch

    rows = sum(n for _, n in segments) + int(np.prod(grid))
    width = heads * 128
    src, inverse, lengths, prefix = H.vsa_plan(segments, rows, *grid)
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
    assert np.array_equal(got[64 * prefix:][live[64 * prefix:]].view(np.uint16),
                          want[64 * prefix:][live[64 * prefix:]].view(np.uint16))
    a, w = (x[:64 * prefix][live[:64 * prefix]].astype(np.float64) for x in (got, want))
    # both forms: f16 probabilities (2^-11) against |v| <= 4.5, pair sums in f16 (2^-9) and an f16 result
    assert np.isfinite(a).all()
    assert np.all(np.abs(a - w) <= 2.0 ** -10 * np.abs(w) + 4.5 * 2.0 ** -9), float(np.abs(a - w).max())
    again = torch.empty_like(out)
    vsa.reset()
    vsa.attend(0, q, k, v, again)
    torch.cuda.synchronize()
    assert torch.equal(out, again)
