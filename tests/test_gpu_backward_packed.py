"""The backward over ragged grids, where the real rows of a chunk come first and halves of 32 slots without any are left out."""
import math

import pytest
import torch

from oracle import bsa_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("keep", [True, False])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("lq,chunk", [
    ((5, 4, 4), (4, 4, 4)),        # two blocks, one of them half a tile: three halves, an odd number
    ((1, 3, 5), (4, 4, 4)),        # every block one half: lists of one or two
    ((6, 9, 13), (4, 4, 4)),       # 32, 16 and 8 rows in the last blocks
    ((5, 8, 13), (4, 4, 8)),       # 80 rows in two tiles, tiles without rows
    ((9, 10, 20), (8, 8, 8)),      # eight tiles a block: more halves than the four bit planes at hand
    ((4, 8, 9), (4, 4, 4)),        # queries and keys padded along one axis alone
])
def test_gradients_on_ragged_grids(lq, chunk, dtype, keep, monkeypatch):
    """Against autograd through fp32 masked-dense attention over the operator's own selection, every block a chunk: P, dS and the
    results are rounded once each (2^-8, 2^-11 relative), so a gradient's 2-norm is off by less than four of those."""
    from longcat_video_amd.block_sparse_attention import bsa_interface as bi
    B, H, S, n = 2, 2, math.prod(lq), math.prod(chunk)
    g = torch.Generator().manual_seed(51)
    q, k, v, do = (torch.randn(B, H, S, 128, generator=g).to(dtype) for _ in range(4))
    dev = [t.cuda() for t in (q, k, v, do)]
    if not keep:
        monkeypatch.setattr(bi, "_backward_workspace", lambda need, least, device: torch.empty(least, dtype=torch.uint8, device=device))
    o, walk, lens, lse = bi._bsa_3d(*dev[:3], lq, lq, 0.4, chunk, chunk, for_backward=True)
    got = bi._bsa_3d_backward(dev[3], *dev[:3], o, lse, walk, lens, lq, lq, chunk, chunk, 128 ** -0.5)
    qp, kp, vp, dop = (O.rearrange_thw_to_3d_block(t, lq, chunk) for t in (q, k, v, do))
    mask = O.block_mask_from_indices(walk.cpu().long(), lens.cpu(), kp.shape[2] // n)
    valid = torch.from_numpy(O.slot_validity(lq, chunk))
    want = O.masked_dense_attention_autograd(qp, kp, vp, dop, mask, n, n, 1 / math.sqrt(128), key_valid=valid)
    ulp = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    for a, w, name in zip(got, want, ("dq", "dk", "dv")):
        w = O.rearrange_3d_block_to_thw(w, lq, chunk).float()
        err = (a.cpu().float() - w).norm() / w.norm()
        assert torch.isfinite(a.float()).all() and float(err) <= 4 * ulp, (name, float(err))
