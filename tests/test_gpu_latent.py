"""GPU: the D = 576 latent attention kernel at the edges of its tiles, pipeline and softmax.

``csa2_attn.fwd`` against the same attention in float64: entry counts around the 32-entry
tiles and the two-step loop (1, 2, 3 tiles and an odd or even number of steps), head counts
around the 64-head workgroup, lists that are not in the top-k's form (empty slots first and
between), and scores that rise so far above the first tile's that the workgroup starts over
from the true maxima.

Bounds: bf16 has 8 significant bits, so a weight is off by at most 2^-8 of itself and the output
by 2^-8 max|v|, and its own rounding adds as much: 2^-7 max|v| (x 1.1 for the float32 sums).  The log-sum-exp is
float32 of scores summed over 576 products: 2^-20 of the largest score's size.
"""

import pytest
import torch

from mzoo_amd import csa2_attn

pytestmark = pytest.mark.gpu


def _reference(q, kv, main, idx, window, sinks):
    b, s, h, d = q.shape
    out, lse = torch.empty(b, s, h, d, dtype=torch.float64), torch.empty(b, h, s, dtype=torch.float64)
    for i in range(b):
        for t in range(s):
            sel = idx[i, t][(idx[i, t] >= 0) & (idx[i, t] < main.shape[1])]
            e = torch.cat([kv[i, max(0, t - window + 1):t + 1, 0], main[i, sel, 0]]).double()
            sc = q[i, t].double() @ e.t() * d ** -0.5
            z = torch.logsumexp(torch.cat([sc, sinks.double()[:, None]], 1), 1)
            out[i, t], lse[i, :, t] = torch.exp(sc - z[:, None]) @ e, z
    return out, lse


def _check(q, kv, main, idx, window, sinks):
    print(f"latent: {tuple(q.shape)} main {main.shape[1]} topk {idx.shape[2]} window {window}", flush=True)
    args = [t.cuda() for t in (q, kv, main, idx)]
    o, lse = csa2_attn.fwd(*args, window=window, compress_ratio=4, sinks=sinks.cuda())
    torch.cuda.synchronize()
    ref, ref_lse = _reference(q, kv, main, idx, window, sinks)
    top = max(kv.abs().max().item(), main.abs().max().item() if main.numel() else 0.0)
    assert (o.cpu().double() - ref).abs().max().item() <= 1.1 * 2.0 ** -7 * top
    size = ref_lse.abs().max().item() + 1.0
    assert (lse.cpu().double() - ref_lse).abs().max().item() <= 2.0 ** -20 * size * 4


def _inputs(seed, heads, topk, groups, seq=3):
    g = torch.Generator().manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    q, kv = rnd(1, seq, heads, 576).bfloat16(), rnd(1, seq, 1, 576).bfloat16()
    main = rnd(1, groups, 1, 576).bfloat16()
    idx = torch.stack([torch.randperm(groups, generator=g)[:topk].sort().values for _ in range(seq)])[None].int()
    return q, kv, main, idx, rnd(heads)


@pytest.mark.parametrize("heads", [1, 17, 64, 65, 128])
@pytest.mark.parametrize("topk", [1, 29, 30, 61, 62, 63, 95, 126, 160])
def test_tile_and_head_edges(heads, topk):
    q, kv, main, idx, sinks = _inputs(topk * 131 + heads, heads, topk, 200)
    _check(q, kv, main, idx, 2, sinks)


@pytest.mark.parametrize("topk", [64, 100, 2052])
def test_lists_with_empty_slots(topk):
    """-1 and out-of-range slots first, between and last; 2052 is read from memory, not ahead."""
    q, kv, main, idx, sinks = _inputs(topk, 20, min(topk, 150), 150)
    pad = torch.full((1, 3, topk), -1, dtype=torch.int32)
    pad[..., :idx.shape[2]] = idx
    pad[:, 0, :40] = -1
    pad[:, 1, 1::2] = 1000
    pad[:, 2, 50:] = -1
    _check(q, kv, main, pad, 1, sinks)


@pytest.mark.parametrize("rise", [1.0, 3.0, 3.7, 12.0])
def test_scores_far_above_the_first_tile(rise):
    """Late entries along head 5's query: its scores rise about 24 * rise nats above the window's
    (84 and more start the workgroup over)."""
    q, kv, main, idx, sinks = _inputs(7, 70, 90, 120)
    main[0, 100:, 0] = (rise * q[0, 1, 5].float()).bfloat16()
    _check(q, kv, main, idx, 2, sinks)
