"""The walk over 32-key halves of a padded grid against the walk over whole blocks."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("latent,chunk,heads,sparsity", [
    ((5, 9, 13), (4, 4, 4), 2, 0.5),        # ragged in every axis; tiles with 1 to 64 keys
    ((4, 6, 8), (4, 4, 4), 1, 0.5),         # halves exactly full: no half of an edge tile but the first
    ((4, 5, 6), (4, 4, 4), 3, 0.25),        # odd numbers of halves
    ((13, 10, 11), (4, 4, 8), 2, 0.5),      # 128-slot chunks with tiles of padding only
    ((5, 9, 20), (2, 8, 16), 2, 0.5),       # 256-slot chunks
    ((9, 34, 61), (4, 4, 4), 7, 0.125),     # several rounds of long lists (337 of 432 blocks: beyond the small list buffers)
])
def test_halves_give_the_bits_of_whole_blocks(dtype, latent, chunk, heads, sparsity):
    """bsa_fwd_3d walks the halves that hold keys, ThwAttention the blocks of the caller's lists with the empty halves
    masked.  A masked half adds zeros, so the outputs agree bit for bit (lists too short to be split over wavefronts, or
    calls of more items than one round)."""
    from longcat_video_amd.block_sparse_attention import bsa_interface as bi
    S = math.prod(latent)
    g = torch.Generator(device="cuda").manual_seed(17)
    q, k, v = (torch.randn(1, heads, S, 128, generator=g, device="cuda").to(dtype) for _ in range(3))
    o, idx, lens, _ = bi._bsa_3d(q, k, v, latent, latent, sparsity, chunk, chunk, want_selection=True)
    nbk = math.prod(-(-n // c) for n, c in zip(latent, chunk))
    paced = bi.visit_order(idx.sort(dim=-1).values.int().contiguous(), lens, nbk)
    assert torch.isfinite(o.float()).all()
    assert torch.equal(bi.ThwAttention(k, v, latent, latent, chunk, chunk)(q, paced, lens), o)
