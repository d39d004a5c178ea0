"""Work items of the attention kernel that several wavefronts of a workgroup share, against one wavefront an item."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("latent,chunk,width", [
    ((4, 4, 8), (4, 4, 4), 2),           # two items: lists of 0, 1 and 2 tiles
    ((5, 9, 13), (4, 4, 4), 5),          # shares of one tile and of two, padded tiles among them
    ((5, 9, 20), (2, 8, 16), 3),         # blocks of four tiles, some of padding alone
    ((13, 10, 11), (4, 4, 8), 20),       # blocks of two tiles
    ((8, 16, 40), (4, 4, 4), 71),        # 80 items: more entries than a wavefront has lanes
    ((8, 34, 40), (4, 4, 4), 180),       # 180 items and lists beyond the small buffers
])
def test_teams_equal_single_wavefronts(dtype, latent, chunk, width):
    """The heads of a call of few items (teams of two and of four) and the same heads among so many that every item has one
    wavefront, over caller's lists of 0 to `width` blocks.  Two orders of the same fp32 sums and two roundings of P: max-abs
    1.6e-2 and mean-abs 1e-3 of outputs near 1, lse 2e-3."""
    from longcat_video_amd.block_sparse_attention import bsa_interface as bi
    S = math.prod(latent)
    blocks = math.prod(-(-n // c) for n, c in zip(latent, chunk))
    tiles = math.prod(chunk) // 64
    g = torch.Generator(device="cuda").manual_seed(21)
    for few in (1, max(1, 300 // (blocks * tiles))):              # up to 256 items a team of four, up to 512 one of two
        q, k, v = (torch.randn(1, few, S, 128, generator=g, device="cuda").to(dtype) for _ in range(3))
        walk = torch.rand(1, few, blocks, blocks, generator=g, device="cuda").argsort(dim=-1)[..., :width].int().contiguous()
        lens = torch.randint(0, width + 1, (1, few, blocks), generator=g, device="cuda", dtype=torch.int32)
        many = -(-1100 // (few * blocks))
        got, lse = bi.ThwAttention(k, v, latent, latent, chunk, chunk)(q, walk, lens, return_lse=True)
        rep = lambda x: x.repeat(1, many, *([1] * (x.dim() - 2)))      # noqa: E731
        want, want_lse = bi.ThwAttention(rep(k), rep(v), latent, latent, chunk, chunk)(rep(q), rep(walk), rep(lens), return_lse=True)
        want, want_lse = want[:, :few], want_lse[:, :few]
        d = (got.float() - want.float()).abs()
        assert d.max() <= 1.6e-2 and d.mean() <= 1e-3, (float(d.max()), float(d.mean()))
        assert torch.equal(torch.isinf(lse), torch.isinf(want_lse))
        assert (lse - want_lse).nan_to_num().abs().max() <= 2e-3


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("heads,sparsity,split", [(9, 0.5, (1152, 128, 4, 1)), (9, 0.75, (1152, 128, 4, 1)), (11, 0.5, (1408, 384, 2, 1))])
def test_last_round_in_teams(heads, sparsity, split, dtype):
    """The items behind whole rounds in teams, against the kernel on whole lists (ThwAttention, which cuts nothing there): the same
    bits in the whole rounds, two summation orders behind them (max-abs 1.6e-2, mean-abs 1e-3, lse 2e-3)."""
    import ctypes
    from longcat_video_amd import _capi
    from longcat_video_amd.block_sparse_attention import bsa_interface as bi
    latent, chunk = (8, 32, 32), (4, 4, 4)
    S = math.prod(latent)
    g = torch.Generator(device="cuda").manual_seed(22)
    q, k, v = (torch.randn(1, heads, S, 128, generator=g, device="cuda").to(dtype) for _ in range(3))
    how = (ctypes.c_int32 * 4)()
    _capi.check(_capi.load().bsa_fwd_3d_last_round(bi._plan_of(1, heads, 128, bi._code(q), latent, latent, chunk, chunk, sparsity, None).prm, how))
    assert tuple(how) == split
    o, walk, lens, lse = bi._bsa_3d(q, k, v, latent, latent, sparsity, chunk, chunk, for_backward=True)
    want, want_lse = bi.ThwAttention(k, v, latent, latent, chunk, chunk)(q, walk, lens, return_lse=True)
    assert torch.equal(o[:, :8], want[:, :8]) and torch.equal(lse[:, :8], want_lse[:, :8])
    d = (o.float() - want.float()).abs()
    assert d.max() <= 1.6e-2 and d.mean() <= 1e-3, (float(d.max()), float(d.mean()))
    assert torch.allclose(lse, want_lse, atol=2e-3)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("latent,chunk,width", [
    ((4, 4, 8), (4, 4, 4), 2),           # two blocks: dQ's lists of one entry, and empty ones, are shared (dK / dV's are too short)
    ((5, 9, 13), (4, 4, 4), 9),          # ragged: tiles of one half, an odd number of halves
    ((13, 10, 11), (4, 4, 8), 20),       # blocks of two tiles, tiles without rows
    ((8, 32, 32), (4, 4, 4), 100),       # 128 tiles, more entries than lanes
])
def test_shared_gradient_lists(latent, chunk, width, dtype):
    """dQ by teams of two and four wavefronts and dK / dV by two pairs of them, against the same heads among so many that every tile
    has its own: the same P and dS, fp32 sums in two orders.  These differ by some 2^-22 of the sum, so one element in
    thousands rounds the other way and the 2-norms differ by far less than an eighth of a rounding."""
    from longcat_video_amd.block_sparse_attention import bsa_interface as bi
    S = math.prod(latent)
    blocks = math.prod(-(-n // c) for n, c in zip(latent, chunk))
    tiles = math.prod(chunk) // 64
    ulp = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    g = torch.Generator(device="cuda").manual_seed(23)
    for few in (1, max(1, 250 // (blocks * tiles)), max(1, 500 // (blocks * tiles))):
        q, k, v, do = (torch.randn(1, few, S, 128, generator=g, device="cuda").to(dtype) for _ in range(4))
        walk = torch.rand(1, few, blocks, blocks, generator=g, device="cuda").argsort(dim=-1)[..., :width].sort(dim=-1).values.int().contiguous()
        lens = torch.randint(0, width + 1, (1, few, blocks), generator=g, device="cuda", dtype=torch.int32)
        o, lse = bi.ThwAttention(k, v, latent, latent, chunk, chunk)(q, walk, lens, return_lse=True)
        args = (latent, latent, chunk, chunk, 128 ** -0.5)
        got = bi._bsa_3d_backward(do, q, k, v, o, lse, walk, lens, *args)
        many = -(-1100 // (few * blocks))
        rep = [x.repeat(1, many, *([1] * (x.dim() - 2))) for x in (do, q, k, v, o, lse, walk, lens)]
        for a, w in zip(got, bi._bsa_3d_backward(*rep, *args)):
            w = w[:, :few].float()
            assert torch.isfinite(a.float()).all()
            assert float((a.float() - w).norm()) <= ulp / 8 * float(w.norm())


@pytest.mark.parametrize("keep", [True, False])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("latent", [(4, 4, 32), (4, 4, 30), (3, 3, 30)])      # eight blocks: full, one of two columns, of one half each
def test_gradient_lists_of_none_one_and_two(latent, dtype, keep, monkeypatch):
    """Lists by hand, 8 x 4 entries for 8 KV blocks, which two pairs of wavefronts share: KV block 0 is listed by one query block,
    so that one pair has nothing, block 1 by none, block 2 by two and the last, which may be ragged, by one.  Bounds as above."""
    from longcat_video_amd.block_sparse_attention import bsa_interface as bi
    chunk, S = (4, 4, 4), math.prod(latent)
    ulp = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    if not keep:
        monkeypatch.setattr(bi, "_backward_workspace", lambda need, least, device: torch.empty(least, dtype=torch.uint8, device=device))
    lists = [[0, 3, 4, 5], [2, 3, 4, 6], [2, 4, 5, 6], [3, 4], [3, 5, 6], [4, 5, 6, 7], [3], []]
    g = torch.Generator(device="cuda").manual_seed(24)
    q, k, v, do = (torch.randn(1, 2, S, 128, generator=g, device="cuda").to(dtype) for _ in range(4))
    walk = torch.tensor([x + [0] * (4 - len(x)) for x in lists], dtype=torch.int32, device="cuda").expand(1, 2, 8, 4).contiguous()
    lens = torch.tensor([len(x) for x in lists], dtype=torch.int32, device="cuda").expand(1, 2, 8).contiguous()
    o, lse = bi.ThwAttention(k, v, latent, latent, chunk, chunk)(q, walk, lens, return_lse=True)
    args = (latent, latent, chunk, chunk, 128 ** -0.5)
    got = bi._bsa_3d_backward(do, q, k, v, o, lse, walk, lens, *args)
    rep = [x.repeat(1, 70, *([1] * (x.dim() - 2))) for x in (do, q, k, v, o, lse, walk, lens)]      # 1 120 tiles: none is shared
    for a, w in zip(got, bi._bsa_3d_backward(*rep, *args)):
        w = w[:, :2].float()
        assert torch.isfinite(a.float()).all()
        assert float((a.float() - w).norm()) <= ulp / 8 * float(w.norm())
    # block 1 is tokens 4 .. 7 of every row: listed by none, its gradients are zero
    column = torch.arange(S, device="cuda") % latent[2]
    for a in got[1:]:
        assert (a[:, :, (column >= 4) & (column < 8)] == 0).all()
