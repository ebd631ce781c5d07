"""GPU: the D = 576 latent attention kernel at the edges of its tiles, pipeline and softmax.

``csa2_attn.fwd`` (bf16 entries) and ``sparse_mqa_decode`` (FP8 entries, one split) against the
same attention in float64: entry counts around the 32-entry tiles and the two-step loop (1, 2, 3
tiles and an odd or even number of steps), head counts around the 64-head workgroup, lists that
are not in the top-k's form (empty slots first and between) and lists that are read ahead or from
memory, scores that rise so far above the first tile's that the workgroup starts over from
the true maxima, and values at both ends of bf16's range.

Bounds, element by element, with A = sum_e w_e |v_e|: a weight is rounded to bf16 (2^-8 of itself,
2^-8 A in the sum) and so is the output (2^-8 |o|); a score s, float32 over 576 products of bf16,
is off by 2^-20 (|s| + the largest |s|) at most, which moves its weight by as much of itself
and the sum by twice that; the float32 sums add 2^-16 A.  The log-sum-exp has the scores'
error alone.  A few percent of slack cover the products of these.
"""

import pytest
import torch

from mzoo_amd import csa2_attn, quant
from oracle import quant as OQ

pytestmark = pytest.mark.gpu
D = 576


def _attend(q, e, sinks):
    """float64: out [H, D], lse [H], A [H, D], the largest |score|."""
    e = e.double()
    sc = q.double() @ e.t() * D ** -0.5
    z = torch.logsumexp(torch.cat([sc, sinks.double()[:, None]], 1), 1)
    w = torch.exp(sc - z[:, None])
    return w @ e, z, w @ e.abs(), sc.abs().max().item()


def _close(o, lse, ref, what):
    out, z, a, top = ref
    sc = 2.0 ** -20 * 2 * (top + 1.0)
    err = (o.double() - out).abs()
    bound = 1.05 * ((2.0 ** -8 + 2.0 ** -16 + 2 * sc) * a + 2.0 ** -8 * out.abs())
    worst = (err / bound.clamp_min(1e-300)).max().item()
    assert bool((err <= bound).all()), f"{what}: output off by {worst:.2f} of its bound"
    assert (lse.double() - z).abs().max().item() <= 1.05 * sc, f"{what}: lse"


def _rows(q, kv, main, idx, window):
    for t in range(q.shape[1]):
        sel = idx[0, t][(idx[0, t] >= 0) & (idx[0, t] < main.shape[1])].long()
        yield t, torch.cat([kv[0, max(0, t - window + 1):t + 1, 0], main[0, sel, 0]])


def _check(q, kv, main, idx, window, sinks):
    """bf16 entries: every row of the prompt."""
    print(f"latent bf16: {tuple(q.shape)} main {main.shape[1]} topk {idx.shape[2]} window {window}", flush=True)
    args = [t.cuda() for t in (q, kv, main, idx)]
    o, lse = (t.cpu() for t in csa2_attn.fwd(*args, window=window, compress_ratio=4, sinks=sinks.cuda()))
    for t, e in _rows(q, kv, main, idx, window):
        _close(o[0, t], lse[0, :, t], _attend(q[0, t], e, sinks), f"row {t}")
    return o, lse


def _check_fp8(q, kv, main, idx, window, sinks):
    """FP8 entries: the prompt's rows as rows of a decode step, each with its own window."""
    s = q.shape[1]
    print(f"latent fp8: {tuple(q.shape)} main {main.shape[1]} topk {idx.shape[2]} window {window}", flush=True)
    win = torch.zeros(s, window, D, dtype=torch.bfloat16)
    for t in range(s):
        for tok in range(max(0, t - window + 1), t + 1):
            win[t, tok % window] = kv[0, tok, 0]
    win_c = quant.pack_latent_fp8_b128(win.cuda())
    main_c = quant.pack_latent_fp8_b128(main[:, :, 0].cuda()).expand(s, -1, -1).contiguous()
    o, lse = csa2_attn.sparse_mqa_decode(q[0].cuda(), torch.arange(s).cuda(), win_c, window, main_cache=main_c,
                                         groups=main.shape[1], indices=idx[0].cuda(), sinks=sinks.cuda(), nsplit=1)
    wu, mu = (torch.from_numpy(OQ.unpack_latent_fp8_b128(c.cpu().numpy())) for c in (win_c, main_c))
    for t in range(s):
        sel = idx[0, t][(idx[0, t] >= 0) & (idx[0, t] < main.shape[1])].long()
        e = torch.cat([wu[t, [tok % window for tok in range(max(0, t - window + 1), t + 1)]], mu[t, sel]])
        _close(o[t].cpu(), lse[t].cpu(), _attend(q[0, t], e, sinks), f"row {t}")


CHECKS = {"bf16": _check, "fp8": _check_fp8}


def _inputs(seed, heads, topk, groups, seq=3):
    g = torch.Generator().manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    q, kv = rnd(1, seq, heads, D).bfloat16(), rnd(1, seq, 1, D).bfloat16()
    main = rnd(1, groups, 1, D).bfloat16()
    idx = torch.stack([torch.randperm(groups, generator=g)[:topk].sort().values for _ in range(seq)])[None].int()
    return q, kv, main, idx, rnd(heads)


@pytest.mark.parametrize("fmt", CHECKS)
@pytest.mark.parametrize("heads", [1, 17, 64, 65, 128])
@pytest.mark.parametrize("topk", [1, 29, 30, 61, 62, 63, 95, 126, 160])
def test_tile_and_head_edges(fmt, heads, topk):
    q, kv, main, idx, sinks = _inputs(topk * 131 + heads, heads, topk, 200)
    CHECKS[fmt](q, kv, main, idx, 2, sinks)


def _with_empty_slots(topk):
    q, kv, main, idx, sinks = _inputs(topk, 20, min(topk, 150), 150)
    pad = torch.full((1, 3, topk), -1, dtype=torch.int32)
    pad[..., :idx.shape[2]] = idx
    pad[:, 0, :40] = -1
    pad[:, 1, 1::2] = 1000
    pad[:, 2, 50:] = -1
    return q, kv, main, pad, sinks


@pytest.mark.parametrize("fmt", CHECKS)
@pytest.mark.parametrize("topk", [64, 100, 2048, 2052])
def test_lists_with_empty_slots(fmt, topk):
    """-1 and out-of-range slots first, between and last; 2052 is read from memory, not ahead."""
    q, kv, main, pad, sinks = _with_empty_slots(topk)
    CHECKS[fmt](q, kv, main, pad, 1, sinks)


@pytest.mark.parametrize("channel", [7, 500, 570])
@pytest.mark.parametrize("topk", [64, 100])
def test_empty_slots_read_no_foreign_entry(topk, channel):
    """An empty slot's place is filled with an entry that the row sees anyway.  Entries outside
    every list are NaN: they reach nothing.  Token 0, the first window entry of rows 0 and 1 (so
    what their empty slots are filled with), is infinite in one channel: each of their heads has
    what float64 gives -- NaN in that channel where its score is -inf, NaN throughout where it
    is +inf -- and row 2, which does not see it, is untouched."""
    q, kv, main, pad, sinks = _with_empty_slots(topk)
    used = torch.unique(pad[(pad >= 0) & (pad < main.shape[1])]).long()
    lone = torch.ones(main.shape[1], dtype=torch.bool)
    lone[used] = False
    main[0, lone] = float("nan")
    _check(q, kv, main, pad, 2, sinks)
    kv[0, 0, 0, channel] = float("inf")
    o, _ = csa2_attn.fwd(*(t.cuda() for t in (q, kv, main, pad)), window=2, compress_ratio=4, sinks=sinks.cuda())
    o = o.cpu()
    for t, e in _rows(q, kv, main, pad, 2):
        want = _attend(q[0, t], e, sinks)[0]
        assert torch.equal(o[0, t].isnan(), want.isnan()), f"row {t}"
        assert bool(want.isnan().any()) == (t < 2)
        fin = ~want.isnan()
        assert (o[0, t].double()[fin] - want[fin]).abs().max().item() <= 2.0 ** -7 * 5


@pytest.mark.parametrize("fmt", CHECKS)
@pytest.mark.parametrize("rise", [1.0, 3.0, 3.7, 12.0])
def test_scores_far_above_the_first_tile(fmt, rise):
    """Late entries along head 5's query: its scores rise about 24 * rise nats above the window's
    (70 and more start the workgroup over)."""
    q, kv, main, idx, sinks = _inputs(7, 70, 90, 120)
    main[0, 100:, 0] = (rise * q[0, 1, 5].float()).bfloat16()
    CHECKS[fmt](q, kv, main, idx, 2, sinks)


@pytest.mark.parametrize("fmt", CHECKS)
@pytest.mark.parametrize("rise,exponent", [(0, -118), (4, -118), (30, -118), (20, 110), (60, 100), (95, 70), (110, 50),
                                           (7, 110), (99, 20)])
def test_values_at_the_ends_of_the_range(fmt, rise, exponent):
    """Entries whose values are about 2^exponent while their scores come from channel 0 alone; the
    last 20 of the list lie 2^rise above the others.  Sums of weights times values leave
    float32's range at either end unless the weights are near 1 (a workgroup that finds
    its sums overflowed starts over from the true maxima)."""
    q, kv, main, idx, sinks = _inputs(rise + 200 + exponent, 3, 120, 120)
    for t in (kv, main):
        t.copy_(torch.ldexp(t.float(), torch.tensor(exponent)))
        t[..., :128] = 0
    q.zero_()
    q[..., 0] = torch.tensor([64.0, 62.0, 60.0])
    main[0, 100:, 0, 0] = rise * 24 / (60 * 1.4426950408889634)
    sinks.fill_(-5.0)
    CHECKS[fmt](q, kv, main, idx, 2, sinks)
