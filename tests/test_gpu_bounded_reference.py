"""The attention kernel without row maxima on items whose norm bound lies above the level that the first keys set: the
fixed reference moves up with the bound, or the item is left to the kernel that looks at the maxima."""
import math

import pytest
import torch

from oracle import bsa_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,scale", [
    (torch.bfloat16, 1.0),      # within the headroom: the reference stays
    (torch.bfloat16, 2.0),      # some 16 (log2) above it
    (torch.bfloat16, 4.0),      # at the far end: items on both sides of the line
    (torch.float16, 0.6),       # fp16 looks at the maxima, whatever the bound
    (torch.float16, 0.9),
    (torch.float16, 1.2),
])
def test_reference_above_the_first_maximum(dtype, scale):
    """1 280 items (two rounds, so the form without maxima runs), lists that start with a tile of masked keys for every
    seventh block.  Against the masked-dense oracle on sampled blocks: the tolerances of the other attention tests
    (max-abs 2e-2 / mean-abs 2e-3, lse 2e-3)."""
    from longcat_video_amd.block_sparse_attention import bsa_interface as bi
    H, nbq, nbk, width = 5, 256, 64, 5
    g = torch.Generator().manual_seed(81)
    q = (torch.randn(1, H, nbq * 64, 128, generator=g) * scale).to(dtype)
    k, v = (torch.randn(1, H, nbk * 64, 128, generator=g).to(dtype) for _ in range(2))
    idx = torch.stack([torch.randperm(nbk, generator=g)[:width].sort().values for _ in range(H * nbq)]).view(1, H, nbq, width).int()
    lens = torch.full((1, H, nbq), width, dtype=torch.int32)
    valid = torch.ones(nbk * 64, dtype=torch.bool)
    valid.view(nbk, 64)[::7, :40] = False                     # a first half without any key
    bits = valid.view(nbk, 64).long().mul(1 << torch.arange(64)).sum(1).cuda()
    o, lse = (t.cpu() for t in bi.attn_fwd_bsa_varlen(q.cuda(), k.cuda(), v.cuda(), 1 / math.sqrt(128), idx.cuda(), lens.cuda(), 64, 64,
                                                      tile_valid=bits, kernel="fragment"))
    assert torch.isfinite(o.float()).all()
    for h, m in ((0, 0), (1, 17), (2, 100), (3, 203), (4, 255)):
        rows = slice(64 * m, 64 * m + 64)
        mask = O.block_mask_from_indices(idx[:, h:h + 1, m:m + 1].long(), lens[:, h:h + 1, m:m + 1], nbk)
        want, want_lse = O.masked_dense_attention(q[:, h:h + 1, rows], k[:, h:h + 1], v[:, h:h + 1], mask, 64, 64, 1 / math.sqrt(128),
                                                  key_valid=valid)
        d = (o[:, h:h + 1, rows].float() - want.float()).abs()
        assert d.max() <= 2e-2 and d.mean() <= 2e-3, (h, m, float(d.max()), float(d.mean()))
        assert torch.allclose(lse[:, h:h + 1, rows], want_lse, rtol=1e-4, atol=2e-3)
