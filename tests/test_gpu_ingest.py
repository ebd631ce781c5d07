"""GPU: a prompt's entries land in the cache slots that the packed caches define.

``append_groups`` and ``fill_window`` take their entry numbers from tables laid out once and
quantize straight into the cache where a row's groups are contiguous; the oracle here is the
quantizer's own output, placed entry by entry.
"""

import pytest
import torch

from mzoo_amd import quant
from mzoo_amd.decode import DecodeConfig, SparseDecodeLayer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt", ["fp8", "mxfp4"])
@pytest.mark.parametrize("b,groups,start,n", [(1, 40, 0, 40), (1, 40, 7, 1), (1, 40, 39, 1), (3, 17, 0, 17), (3, 17, 5, 9)])
def test_append_groups_places_entries(dev, fmt, b, groups, start, n):
    layer = SparseDecodeLayer(DecodeConfig(batch=b, max_groups=groups, index_format=fmt, nsplit=1), dev)
    gen = torch.Generator().manual_seed(b * 100 + n)
    lat = torch.randn(b, n, 576, generator=gen).bfloat16().to(dev)
    keys = torch.randn(b, n, 128, generator=gen).bfloat16().to(dev)
    kc = (layer.k_codes, layer.k_scales) if fmt == "fp8" else (layer.k_packed, layer.k_e8m0)
    want = [t.clone() for t in (layer.main, *kc)]
    layer.append_groups(start, lat, keys)
    q = quant.quant_fp8_block(keys, 128) if fmt == "fp8" else quant.quant_mxfp4(keys)
    q = (q[0], q[1][..., 0]) if fmt == "fp8" else q
    for t, v in zip(want, (quant.pack_latent_fp8_b128(lat), *q)):
        for j in range(n):
            t[:, start + j] = v[:, j]
    assert all(torch.equal(a, w) for a, w in zip((layer.main, *kc), want))
    with pytest.raises((ValueError, RuntimeError)):
        layer.append_groups(groups - 1, lat.new_zeros(b, 2, 576), keys.new_zeros(b, 2, 128))


@pytest.mark.parametrize("b,last", [(1, 127), (1, 128), (3, 200), (2, 255), (2, 5000)])
def test_fill_window_places_tokens(dev, b, last):
    layer = SparseDecodeLayer(DecodeConfig(batch=b, max_groups=8, nsplit=1), dev)
    w = layer.cfg.window
    lat = torch.randn(b, w, 576, generator=torch.Generator().manual_seed(last)).bfloat16().to(dev)
    layer.fill_window(lat, last)
    ent = quant.pack_latent_fp8_b128(lat)
    for j, tok in enumerate(range(last - w + 1, last + 1)):
        assert torch.equal(layer.win.view(b, w, -1)[:, tok % w], ent[:, j])


def test_quantizers_refuse_an_unfit_out(dev):
    x = torch.randn(4, 128).bfloat16().to(dev)
    codes, scales = quant.quant_fp8_block(x)
    for bad in [(codes[:3], scales), (codes, scales.double()), (torch.empty(4, 256, dtype=torch.uint8, device=dev)[:, ::2], scales)]:
        with pytest.raises(ValueError):
            quant.quant_fp8_block(x, out=bad)
    packed, e8 = quant.quant_mxfp4(x)
    with pytest.raises(ValueError):
        quant.quant_mxfp4(x, out=(packed, e8[:2]))
