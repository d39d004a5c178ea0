"""Calls of one round, whose workgroups make the lists that they walk, against the kernels that make them by themselves."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("latent,chunk,heads,sparsity", [
    ((4, 4, 4), (4, 4, 4), 1, 0.0),             # one block
    ((4, 32, 32), (4, 4, 4), 2, 0.9),           # 64 blocks, a team of four, 6 kept: no visiting order
    ((4, 32, 32), (4, 4, 4), 8, 0.8),           # ... 512 items, teams of two
    ((4, 32, 32), (4, 4, 4), 9, 0.8),           # ... 576, one wavefront an item
    ((4, 20, 52), (4, 4, 4), 3, 0.5),           # 65 blocks
    ((8, 32, 32), (4, 4, 4), 8, 0.75),          # 128 blocks, one wavefront an item
    ((4, 12, 172), (4, 4, 4), 7, 0.75),         # 129: more than two columns a lane
    ((16, 32, 32), (4, 4, 4), 4, 0.3),          # 256 blocks, the most a wavefront scores; 179 kept
    ((4, 4, 1028), (4, 4, 4), 3, 0.9),          # 257, 771 items: the kernel in front
    ((8, 64, 64), (4, 4, 4), 1, 0.8),           # 512: the most a team scores
    ((4, 4, 2052), (4, 4, 4), 1, 0.9),          # 513: the kernels in front
    ((5, 9, 13), (4, 4, 4), 2, 0.5),            # ragged: halves
    ((5, 33, 30), (4, 4, 4), 7, 0.7),           # ... 144 blocks, 1 008 items
    ((13, 10, 11), (4, 4, 8), 3, 0.4),          # blocks of two tiles, tiles of padding alone
    ((8, 16, 32), (4, 8, 8), 2, 0.5),           # blocks of four tiles without padding
])
def test_lists_made_by_the_attention_kernel(latent, chunk, heads, sparsity, dtype):
    """The lists that a backward would be given are those of score, top-k and visiting order one after another, with equal scores
    among them (repeated key chunks: ties go to the lowest block), and the output is theirs bit for bit, with and without lists."""
    from longcat_video_amd.block_sparse_attention import bsa_interface as bi
    S, blocks = math.prod(latent), math.prod(-(-n // c) for n, c in zip(latent, chunk))
    g = torch.Generator(device="cuda").manual_seed(31)
    for ties in (False, True):
        q, k, v = (torch.randn(2, heads, S, 128, generator=g, device="cuda").to(dtype)[:1] for _ in range(3))
        if ties:
            k[:, :, S // 2:] = k[:, :, :1]
        o, walk, lens, lse = bi._bsa_3d(q, k, v, latent, latent, sparsity, chunk, chunk, for_backward=True)
        want_o, idx, want_lens, _ = bi._bsa_3d(q, k, v, latent, latent, sparsity, chunk, chunk, want_selection=True)
        ascending = idx.sort(dim=-1).values.int().contiguous()
        assert torch.equal(lens, want_lens) and torch.equal(walk, bi.visit_order(ascending, lens, blocks))
        assert torch.isfinite(o.float()).all() and torch.equal(o, want_o)
        assert torch.equal(bi.flash_attn_bsa_3d(q, k, v, latent, latent, sparsity=sparsity, chunk_3d_shape_q=chunk, chunk_3d_shape_k=chunk), o)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("latent,chunk,heads,threshold,sparsity", [
    ((4, 4, 4), (4, 4, 4), 1, 0.5, None),             # one block, which alone is more than the threshold: an empty list
    ((4, 32, 32), (4, 4, 4), 2, 0.5, None),           # a team of four
    ((4, 32, 32), (4, 4, 4), 9, 0.25, 0.9),           # one wavefront an item, never fewer than six blocks
    ((16, 32, 32), (4, 4, 4), 1, 1.0, None),          # every one of 256 blocks
    ((5, 9, 13), (4, 4, 4), 2, 0.75, 0.5),            # ragged: halves
    ((13, 10, 11), (4, 4, 8), 3, 0.5, None),          # blocks of two tiles, tiles of padding alone
    ((8, 32, 36), (4, 4, 4), 8, 0.5, None),           # 1 152 items: the kernels in front
])
def test_cdf_lists_made_by_the_attention_kernel(latent, chunk, heads, threshold, sparsity, dtype):
    """The same for the CDF rule, with scores that differ in their spread from block to block, with equal ones, and with a NaN
    (its rows keep every block)."""
    from longcat_video_amd.block_sparse_attention import bsa_interface as bi
    S, blocks = math.prod(latent), math.prod(-(-n // c) for n, c in zip(latent, chunk))
    g = torch.Generator(device="cuda").manual_seed(32)
    for kind in ("spread", "ties", "nan"):
        q, k, v = (torch.randn(1, heads, S, 128, generator=g, device="cuda") for _ in range(3))
        k = k + 3 * torch.randn(1, heads, 1, 128, generator=g, device="cuda")
        q = q * torch.rand(1, heads, S, 1, generator=g, device="cuda") * 4
        if kind == "ties":
            k[:, :, S // 2:] = k[:, :, :1]
        q, k, v = (x.to(dtype) for x in (q, k, v))
        if kind == "nan":
            q[0, 0, 0, 0] = float("nan")
        args = (q, k, v, latent, latent, sparsity, chunk, chunk)
        o, walk, lens, _ = bi._bsa_3d(*args, for_backward=True, cdf_threshold=threshold)
        want_o, idx, want_lens, _ = bi._bsa_3d(*args, want_selection=True, cdf_threshold=threshold)
        ascending = torch.where(idx < 0, torch.full_like(idx, blocks), idx).sort(dim=-1).values
        want = bi.visit_order(torch.where(ascending == blocks, torch.zeros_like(ascending), ascending).int(), want_lens, blocks)
        used = torch.arange(blocks, device="cuda") < want_lens[..., None]
        assert torch.equal(lens, want_lens) and torch.equal(walk[used], want[used]) and (walk[~used] == -1).all()
        assert torch.equal(o.nan_to_num(), want_o.nan_to_num()) and torch.equal(o.isnan(), want_o.isnan())


@pytest.mark.parametrize("latent,chunk,heads,sparsity", [
    ((4, 4, 4), (4, 4, 4), 1, 0.0),
    ((4, 8, 8), (4, 4, 4), 4, 0.5),
    ((4, 32, 32), (4, 4, 4), 4, 0.9),           # 64 blocks, 1 024 units: the most
    ((4, 20, 52), (4, 4, 4), 2, 0.5),           # 65
    ((8, 32, 32), (4, 4, 4), 1, 0.75),          # 128: the most
    ((4, 12, 172), (4, 4, 4), 1, 0.75),         # 129: the kernel in front
    ((5, 9, 13), (4, 4, 4), 2, 0.5),            # ragged
    ((13, 10, 11), (4, 4, 8), 1, 0.4),          # blocks of eight units, some of padding alone
])
def test_fp32_lists_made_by_the_attention_kernel(latent, chunk, heads, sparsity):
    """The same for fp32 operands, by the output alone: another list would be another output."""
    from longcat_video_amd.block_sparse_attention import bsa_interface as bi
    S = math.prod(latent)
    g = torch.Generator(device="cuda").manual_seed(33)
    for ties in (False, True):
        q, k, v = (torch.randn(2, heads, S, 128, generator=g, device="cuda")[:1] for _ in range(3))
        if ties:
            k[:, :, S // 2:] = k[:, :, :1]
        want = bi._bsa_3d(q, k, v, latent, latent, sparsity, chunk, chunk, want_selection=True)[0]
        got = bi.flash_attn_bsa_3d(q, k, v, latent, latent, sparsity=sparsity, chunk_3d_shape_q=chunk, chunk_3d_shape_k=chunk)
        assert torch.isfinite(got).all() and torch.equal(got, want)


def _unlike(kind, big, latent, q, k):
    """q and k, fp32, with scores among them that are infinite or no number."""
    if kind == "inf":                               # the columns of blocks at both edges: scores of both signs beyond the storage type
        w = torch.arange(q.shape[2], device="cuda") % latent[2]
        k[:, :, w < latent[2] // 4, 0] = big
        k[:, :, w >= latent[2] - latent[2] // 4, 0] = -big
        q[..., 0] = 4
    else:
        q[:, 0, 3, 7] = float("nan")                # all scores of a block
        k[:, -1, -2, 5] = float("nan")              # one of every block
        k[:, 0, 1, 6] = -float("nan")
    return q, k


@pytest.mark.parametrize("kind", ["inf", "nan"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("latent,chunk,heads,threshold,sparsity", [
    ((4, 32, 32), (4, 4, 4), 2, None, 0.8),           # teams of four
    ((4, 32, 32), (4, 4, 4), 9, None, 0.5),           # one wavefront an item
    ((4, 12, 172), (4, 4, 4), 2, None, 0.6),
    ((8, 64, 64), (4, 4, 4), 1, None, 0.9),           # eight columns a lane
    ((5, 9, 13), (4, 4, 4), 2, None, 0.5),            # ragged
    ((4, 32, 32), (4, 4, 4), 2, 0.5, None),
    ((4, 32, 32), (4, 4, 4), 9, 0.25, 0.9),
    ((16, 32, 32), (4, 4, 4), 1, 0.75, None),
    ((5, 9, 13), (4, 4, 4), 2, 0.75, 0.5),
])
def test_infinite_scores_and_nan(latent, chunk, heads, threshold, sparsity, dtype, kind):
    """The attention kernel's file is built without regard for NaN: its lists, of rows with infinite scores and with NaN (which
    sorts above them by its bits), are those of the kernels in front all the same."""
    from longcat_video_amd.block_sparse_attention import bsa_interface as bi
    S, blocks = math.prod(latent), math.prod(-(-n // c) for n, c in zip(latent, chunk))
    g = torch.Generator(device="cuda").manual_seed(34)
    q, k, v = (torch.randn(1, heads, S, 128, generator=g, device="cuda") for _ in range(3))
    q, k = _unlike(kind, 3e38 if dtype == torch.bfloat16 else 6e4, latent, q, k)
    args = (q.to(dtype), k.to(dtype), v.to(dtype), latent, latent, sparsity, chunk, chunk)
    o, walk, lens, _ = bi._bsa_3d(*args, for_backward=True, cdf_threshold=threshold)
    want_o, idx, want_lens, score = bi._bsa_3d(*args, want_selection=True, cdf_threshold=threshold)
    assert (score.isinf() if kind == "inf" else score.isnan()).any()
    ascending = torch.where(idx < 0, torch.full_like(idx, blocks), idx).sort(dim=-1).values
    want = bi.visit_order(torch.where(ascending == blocks, torch.zeros_like(ascending), ascending).int().contiguous(), want_lens, blocks)
    used = torch.arange(want.shape[-1], device="cuda") < want_lens[..., None]
    assert torch.equal(lens, want_lens) and torch.equal(walk[used], want[used])
    assert torch.equal(o.isnan(), want_o.isnan()) and torch.equal(o.nan_to_num(), want_o.nan_to_num())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("latent_q,latent_k,chunk_q,chunk_k,batch,heads,threshold,sparsity", [
    ((4, 4, 4), (4, 32, 32), (4, 4, 4), (4, 4, 4), 1, 1, None, 0.5),              # one query block
    ((4, 8, 8), (12, 8, 8), (4, 4, 4), (4, 4, 4), 2, 3, None, 0.5),               # more key frames
    ((12, 8, 8), (4, 8, 8), (4, 4, 4), (4, 4, 4), 3, 2, None, 0.3),               # fewer
    ((4, 32, 32), (4, 16, 32), (4, 4, 4), (4, 4, 8), 2, 5, None, 0.5),            # chunks of different size, 640 items
    ((4, 16, 32), (8, 16, 32), (4, 4, 8), (4, 4, 4), 2, 2, None, 0.7),            # ... query blocks of two tiles
    ((5, 9, 13), (13, 10, 11), (4, 4, 4), (4, 4, 8), 2, 2, None, 0.6),            # ragged on both sides
    ((13, 10, 11), (5, 9, 13), (2, 8, 16), (4, 4, 4), 2, 1, None, 0.4),
    ((4, 8, 8), (12, 8, 8), (4, 4, 4), (4, 4, 4), 2, 3, 0.5, None),
    ((5, 9, 13), (13, 10, 11), (4, 4, 4), (4, 4, 8), 2, 2, 0.5, 0.8),
    ((4, 16, 32), (8, 16, 32), (4, 4, 8), (4, 4, 4), 2, 2, 0.25, None),
])
def test_queries_and_keys_of_different_grids(latent_q, latent_k, chunk_q, chunk_k, batch, heads, threshold, sparsity, dtype):
    """The lists and the output of calls whose queries and keys differ in frames, in extent or in chunks, in batches."""
    from longcat_video_amd.block_sparse_attention import bsa_interface as bi
    blocks = math.prod(-(-n // c) for n, c in zip(latent_k, chunk_k))
    g = torch.Generator(device="cuda").manual_seed(35)
    q = torch.randn(batch, heads, math.prod(latent_q), 128, generator=g, device="cuda").to(dtype)
    k, v = (torch.randn(batch, heads, math.prod(latent_k), 128, generator=g, device="cuda").to(dtype) for _ in range(2))
    args = (q, k, v, latent_q, latent_k, sparsity, chunk_q, chunk_k)
    o, walk, lens, _ = bi._bsa_3d(*args, for_backward=True, cdf_threshold=threshold)
    want_o, idx, want_lens, _ = bi._bsa_3d(*args, want_selection=True, cdf_threshold=threshold)
    ascending = torch.where(idx < 0, torch.full_like(idx, blocks), idx).sort(dim=-1).values
    want = bi.visit_order(torch.where(ascending == blocks, torch.zeros_like(ascending), ascending).int().contiguous(), want_lens, blocks)
    used = torch.arange(want.shape[-1], device="cuda") < want_lens[..., None]
    assert torch.equal(lens, want_lens) and torch.equal(walk[used], want[used])
    assert torch.isfinite(o.float()).all() and torch.equal(o, want_o)
    assert torch.equal(bi.flash_attn_bsa_3d(q, k, v, latent_q, latent_k, sparsity=sparsity, cdf_threshold=threshold,
                                            chunk_3d_shape_q=chunk_q, chunk_3d_shape_k=chunk_k), o)
