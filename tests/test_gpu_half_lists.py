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
    ((13, 10, 11), (4, 4, 8), 2, 0.75),     # 128-slot chunks with tiles of padding only
    ((5, 9, 20), (2, 8, 16), 2, 0.75),      # 256-slot chunks
    ((9, 34, 61), (4, 4, 4), 7, 0.125),     # several rounds of long lists (337 of 432 blocks: beyond the small list buffers)
])
def test_halves_give_the_bits_of_whole_blocks(dtype, latent, chunk, heads, sparsity):
    """bsa_fwd_3d walks the halves that hold keys, ThwAttention the blocks of the caller's lists with the empty halves
    masked.  A masked half adds zeros, so the outputs agree bit for bit.  (Lists under 20 tiles, or no partial round worth
    cutting: a list that is cut into parts rounds differently.)"""
    from longcat_video_amd.block_sparse_attention import bsa_interface as bi
    S = math.prod(latent)
    g = torch.Generator(device="cuda").manual_seed(17)
    q, k, v = (torch.randn(1, heads, S, 128, generator=g, device="cuda").to(dtype) for _ in range(3))
    o, idx, lens, _ = bi._bsa_3d(q, k, v, latent, latent, sparsity, chunk, chunk, want_selection=True)
    nbk = math.prod(-(-n // c) for n, c in zip(latent, chunk))
    paced = bi.visit_order(idx.sort(dim=-1).values.int().contiguous(), lens, nbk)
    assert torch.isfinite(o.float()).all()
    assert torch.equal(bi.ThwAttention(k, v, latent, latent, chunk, chunk)(q, paced, lens), o)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("latent,heads,sparsity", [
    ((4, 12, 44), 1, 0.3),         # 33 items of 23 tiles: two parts
    ((8, 16, 32), 1, 0.25),        # 64 items of 48 tiles: four
    ((9, 33, 30), 1, 0.1),         # 216 items, ragged: parts of different lengths, items of 16 rows
    ((8, 32, 36), 8, 0.5),         # 1 152 items: a whole round, then 128 items in parts
    ((8, 32, 40), 10, 0.5),        # 1 600: 576 left over, which stay whole
])
def test_items_in_parts(dtype, latent, heads, sparsity):
    """A partial round is cut into parts along the lists and merged: against the kernel on whole lists (two summation
    orders: max-abs 1.6e-2, mean-abs 1e-3, lse 2e-3), with and without padded rows."""
    from longcat_video_amd.block_sparse_attention import bsa_interface as bi
    S, chunk = math.prod(latent), (4, 4, 4)
    g = torch.Generator(device="cuda").manual_seed(18)
    q, k, v = (torch.randn(1, heads, S, 128, generator=g, device="cuda").to(dtype) for _ in range(3))
    o, walk, lens, lse = bi._bsa_3d(q, k, v, latent, latent, sparsity, chunk, chunk, for_backward=True)
    want, want_lse = bi.ThwAttention(k, v, latent, latent, chunk, chunk)(q, walk, lens, return_lse=True)
    d = (o.float() - want.float()).abs()
    assert d.max() <= 1.6e-2 and d.mean() <= 1e-3, (float(d.max()), float(d.mean()))
    assert torch.allclose(lse, want_lse, atol=2e-3)
    assert torch.equal(bi.flash_attn_bsa_3d(q, k, v, latent, latent, sparsity=sparsity, chunk_3d_shape_q=chunk, chunk_3d_shape_k=chunk), o)
