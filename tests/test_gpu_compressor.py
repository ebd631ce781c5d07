"""GPU parity of the compressor (piece 2) and RoPE: bit-exact against the CPU oracle.

Both evaluate the same pinned float32 operation sequence (oracle/compressor.py), so every
output bit must match, for fp32 and bf16 models, ratios 1/2/4/128 and the two latent
widths (576 = 512+64, 160 = 128+32).  Also: the group carry across calls
(``store_compression_weights``, owlet1/cache.py:96-113) gives the same latents as one call.
"""

import numpy as np
import pytest
import torch

from mzoo_amd import cache as MC
from oracle import compressor as C

pytestmark = pytest.mark.gpu
NAMES = {torch.float32: "float32", torch.bfloat16: "bfloat16"}


def _bits(t):
    t = t.cpu()
    return t.view(torch.int32).numpy() if t.dtype == torch.float32 else t.view(torch.int16).numpy()


def _obits(x, dtype):
    return _bits(torch.from_numpy(np.ascontiguousarray(x)).to(dtype))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("ratio,d", [(4, 576), (2, 160), (128, 576), (1, 576), (4, 160)])
def test_compress_bit_exact(dev, dtype, ratio, d):
    gen = torch.Generator().manual_seed(ratio * 1000 + d)
    b, n = 3, 40 if ratio < 128 else 3
    kv = torch.randn(b, n * ratio + 1, d, generator=gen)            # one trailing token left over
    gate = torch.randn(b, n * ratio + 1, d, generator=gen) * 4
    w = (1 + 0.1 * torch.randn(d, generator=gen)).to(dtype)
    got = MC.compress(kv.to(dev), gate.to(dev) if ratio > 1 else None, ratio, w.to(dev), 1e-20, dtype, n_groups=n)
    want = C.compress(kv[:, :n * ratio].numpy(), gate[:, :n * ratio].numpy(), ratio, w.float().numpy(), 1e-20,
                      NAMES[dtype])
    assert np.array_equal(_bits(got), _obits(want, dtype))


@pytest.mark.parametrize("ratio,d", [(2, 1), (4, 65), (4, 1024), (2, 1000), (1, 129), (3, 100), (7, 1024), (8, 576),
                                     (9, 64), (130, 1), (17, 65)])
def test_compress_edges_bit_exact(dev, ratio, d):
    """Channel counts around the wave and the two channels a lane loads together (ratios 1, 2,
    4), token counts around the 8 that the other ratios load together; a gate of -inf and one
    far below the maximum take their weights' limits."""
    gen = torch.Generator().manual_seed(ratio * 1000 + d)
    b, n = 2, 5
    kv = torch.randn(b, n * ratio + 1, d, generator=gen)
    gate = torch.randn(b, n * ratio + 1, d, generator=gen) * 30
    if ratio > 1:
        gate[0, 1, d // 2] = float("-inf")
        gate[1, 0, 0] = -200.0
    w = (1 + 0.1 * torch.randn(d, generator=gen)).bfloat16()
    got = MC.compress(kv.to(dev), gate.to(dev) if ratio > 1 else None, ratio, w.to(dev), 1e-20, torch.bfloat16, n_groups=n)
    want = C.compress(kv[:, :n * ratio].numpy(), gate[:, :n * ratio].numpy(), ratio, w.float().numpy(), 1e-20, "bfloat16")
    assert np.array_equal(_bits(got), _obits(want, torch.bfloat16))


def test_compressor_carry_matches_one_shot(dev):
    gen = torch.Generator().manual_seed(9)
    kv = torch.randn(2, 37, 576, generator=gen).to(dev)
    gate = torch.randn(2, 37, 576, generator=gen).to(dev)
    w = torch.ones(576, dtype=torch.bfloat16, device=dev)
    one, first = MC.compressor_forward(kv, gate, 4, w, 1e-20, torch.bfloat16, MC.GroupCarry())
    assert first == 0 and one.shape == (2, 9, 576)
    carry, parts, starts = MC.GroupCarry(), [], []
    for a, z in [(0, 3), (3, 4), (4, 11), (11, 12), (12, 37)]:
        lat, f = MC.compressor_forward(kv[:, a:z], gate[:, a:z], 4, w, 1e-20, torch.bfloat16, carry)
        if lat is not None:
            parts.append(lat)
            starts.append(f)
            carry.emitted(lat.shape[1])
    # tokens 0-3 complete in call 2, 4-7 in call 3, 8-11 in call 4, 12-35 in call 5
    assert starts == [0, 4, 8, 12]
    assert torch.equal(torch.cat(parts, 1), one)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_rope_bit_exact(dev, dtype):
    gen = torch.Generator().manual_seed(3)
    x = torch.randn(2, 9, 4, 576, generator=gen).to(dtype)
    cos, sin = C.rope_tables(np.random.default_rng(0).integers(0, 32768, (2, 9)), 64, 160000.0)
    for inverse in (False, True):
        got = MC.apply_rotary_pos_emb(x.to(dev), torch.from_numpy(cos).to(dev), torch.from_numpy(sin).to(dev),
                                      inverse=inverse)
        want = C.rope(x.float().numpy(), cos[:, :, None], sin[:, :, None], inverse, NAMES[dtype])
        assert np.array_equal(_bits(got), _obits(want, dtype))


@pytest.mark.parametrize("ratio,groups,d", [(3, 1023, 100), (3, 1024, 65), (3, 1025, 1), (5, 1535, 64), (5, 1539, 576),
                                            (3, 1024, 1024)])
def test_compress_forms_of_ratios_3_and_5(dev, ratio, groups, d):
    """On both sides of the line between the workgroup and the wave form: the oracle's bits."""
    gen = torch.Generator().manual_seed(groups + d)
    kv, gate = torch.randn(1, groups * ratio, d, generator=gen), torch.randn(1, groups * ratio, d, generator=gen) * 5
    w = (1 + 0.1 * torch.randn(d, generator=gen)).bfloat16()
    got = MC.compress(kv.to(dev), gate.to(dev), ratio, w.to(dev), 1e-6, torch.bfloat16)
    want = C.compress(kv.numpy(), gate.numpy(), ratio, w.float().numpy(), 1e-6, "bfloat16")
    assert np.array_equal(_bits(got), _obits(want, torch.bfloat16))


def test_compress_more_threads_than_one_grid_axis(dev):
    """From 2^32 threads (here 34 M groups of 65 channels, 128 threads each) the launch takes a
    second grid axis: the groups at both ends and around its turns equal those of small calls.
    One tensor of 52 GB is the projection and the gate, zero but in those groups."""
    d, ratio, n = 65, 6, (1 << 25) + 5
    if torch.cuda.mem_get_info(dev)[0] < (64 << 30):
        pytest.skip("needs 64 GB of GPU memory")
    gen = torch.Generator().manual_seed(3)
    starts = [0, (1 << 21) - 2, (1 << 22) - 2, (1 << 24) - 2, (1 << 25) - 2, n - 2]
    kv = torch.zeros(1, n * ratio, d, device=dev)
    w = (1 + 0.1 * torch.randn(d, generator=gen)).bfloat16().to(dev)
    for g in starts:
        kv[:, g * ratio:(g + 4) * ratio].copy_(torch.randn(1, min(4, n - g) * ratio, d, generator=gen).to(dev))
    out = MC.compress(kv, kv, ratio, w, 1e-6, torch.bfloat16)
    for g in starts:
        part = kv[:, g * ratio:(g + 4) * ratio]
        assert torch.equal(out[:, g:g + 4], MC.compress(part, part, ratio, w, 1e-6, torch.bfloat16)), f"groups {g}.."
