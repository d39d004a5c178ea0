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
@pytest.mark.parametrize("latent_q,latent_k,chunk,heads,sparsity,split", [
    # (work items, items of the last round, wavefronts to a share, shares): teams
    ((4, 12, 44), (4, 12, 44), (4, 4, 4), 1, 0.3, (33, 33, 4, 1)),
    ((8, 16, 32), (8, 16, 32), (4, 4, 4), 1, 0.25, (64, 64, 4, 1)),
    ((9, 33, 30), (9, 33, 30), (4, 4, 4), 1, 0.1, (216, 216, 4, 1)),           # ragged: shares of different lengths, items of 16 rows
    ((8, 32, 36), (8, 32, 36), (4, 4, 4), 8, 0.5, (1152, 128, 4, 1)),          # a whole round in front
    ((8, 32, 40), (8, 32, 40), (4, 4, 4), 10, 0.5, (1600, 576, 1, 1)),         # 576 left over, which stay whole
    # parts, merged by another launch
    ((8, 16, 32), (8, 16, 32), (4, 4, 4), 1, 0.0, (64, 64, 2, 3)),
    ((8, 32, 32), (8, 32, 32), (4, 4, 4), 1, 0.05, (128, 128, 4, 2)),
    ((8, 32, 32), (8, 32, 32), (4, 4, 4), 9, 0.05, (1152, 128, 4, 2)),
    ((8, 32, 32), (8, 32, 32), (4, 4, 4), 10, 0.25, (1280, 256, 2, 2)),
    ((16, 32, 32), (16, 32, 32), (4, 4, 4), 6, 0.5, (1536, 512, 1, 2)),        # a wavefront a part
    ((4, 4, 32), (4, 20, 64), (4, 4, 4), 1, 0.0, (8, 8, 2, 4)),                # few queries
    ((5, 9, 13), (9, 33, 30), (4, 4, 4), 1, 0.25, (24, 24, 2, 8)),             # ... and ragged on both sides
    ((5, 9, 13), (9, 33, 30), (4, 4, 4), 2, 0.07, (48, 48, 4, 5)),
    ((13, 10, 11), (13, 30, 31), (4, 4, 8), 1, 0.5, (30, 30, 2, 6)),           # blocks of two tiles, tiles of padding alone
    ((13, 10, 11), (13, 30, 31), (2, 8, 16), 1, 0.7, (27, 27, 2, 3)),          # of four
])
def test_items_in_parts(dtype, latent_q, latent_k, chunk, heads, sparsity, split):
    """A partial round is shared by teams and cut into parts along the lists: against the same heads among so many that every
    item has one wavefront (two summation orders: max-abs 1.6e-2, mean-abs 1e-3, lse 2e-3), with and without padded rows."""
    import ctypes
    from longcat_video_amd import _capi
    from longcat_video_amd.block_sparse_attention import bsa_interface as bi
    g = torch.Generator(device="cuda").manual_seed(18)
    q = torch.randn(1, heads, math.prod(latent_q), 128, generator=g, device="cuda").to(dtype)
    k, v = (torch.randn(1, heads, math.prod(latent_k), 128, generator=g, device="cuda").to(dtype) for _ in range(2))
    how = (ctypes.c_int32 * 4)()
    plan = bi._plan_of(1, heads, 128, bi._code(q), latent_q, latent_k, chunk, chunk, sparsity, None)
    _capi.check(_capi.load().bsa_fwd_3d_last_round(plan.prm, how))
    assert tuple(how) == split
    o, walk, lens, lse = bi._bsa_3d(q, k, v, latent_q, latent_k, sparsity, chunk, chunk, for_backward=True)
    many = -(-1100 // split[0])
    rep = lambda x: x.repeat(1, many, *([1] * (x.dim() - 2)))      # noqa: E731
    want, want_lse = bi.ThwAttention(rep(k), rep(v), latent_q, latent_k, chunk, chunk)(rep(q), rep(walk), rep(lens), return_lse=True)
    want, want_lse = want[:, :heads], want_lse[:, :heads]
    d = (o.float() - want.float()).abs()
    assert d.max() <= 1.6e-2 and d.mean() <= 1e-3, (float(d.max()), float(d.mean()))
    assert torch.allclose(lse, want_lse, atol=2e-3)
    assert torch.equal(bi.flash_attn_bsa_3d(q, k, v, latent_q, latent_k, sparsity=sparsity, chunk_3d_shape_q=chunk, chunk_3d_shape_k=chunk), o)
