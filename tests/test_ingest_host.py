"""CPU: where ``append_groups`` lets the quantizer write (the quantizers themselves are replaced)."""

import pytest
import torch

from mzoo_amd import quant
from mzoo_amd.decode import DecodeConfig, SparseDecodeLayer


@pytest.mark.parametrize("batch,device,rows,direct", [(1, "cpu", 1, True), (1, "meta", 1, False), (3, "cpu", 3, False),
                                                      (3, "cpu", 1, False)])
def test_append_groups_targets(monkeypatch, batch, device, rows, direct):
    """One row's keys go straight into the cache; several rows' (strided there), one row's for
    all (broadcast) and keys on another device are quantized where they are, then copied."""
    layer = object.__new__(SparseDecodeLayer)
    layer.cfg = DecodeConfig(batch=batch, max_groups=8)
    layer.main = torch.zeros(batch, 8, 656, dtype=torch.uint8)
    layer._group_rows = torch.arange(batch * 8).view(batch, 8)
    layer.k_codes = torch.zeros(batch, 8, 128, dtype=torch.uint8)
    layer.k_scales = torch.zeros(batch, 8)
    seen = []

    def quantize(x, block, out=None):
        seen.append(out is not None)
        codes, scales = out or (torch.empty(*x.shape, dtype=torch.uint8), torch.empty(*x.shape[:-1], 1))
        assert out is None or out[0].device == x.device
        return codes.fill_(7), scales.fill_(3.0)

    monkeypatch.setattr(quant, "pack_latent_fp8_b128", lambda *a, **k: None)
    monkeypatch.setattr(quant, "quant_fp8_block", quantize)
    layer.append_groups(2, torch.zeros(batch, 3, 576), torch.zeros(rows, 3, 128, device=device))
    assert seen == [direct]
    want = torch.zeros(8)
    want[2:5] = 1
    assert torch.equal(layer.k_codes.float(), (7 * want)[None, :, None].expand(batch, 8, 128))
    assert torch.equal(layer.k_scales, (3 * want).expand(batch, 8))
