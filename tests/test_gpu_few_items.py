"""The attention kernel of calls that leave SIMDs idle (32x32x16 products, K and V in their order) against that of calls that do not."""
import ctypes
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

CHUNK = (4, 4, 4)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("heads,latent,sparsity,split", [
    (1, (4, 40, 160), 0.9, (400, 400, 2, 1)),          # 400 items and 401: both sides of the line for teams of two
    (1, (4, 4, 1604), 0.9, (401, 401, 2, 1)),
    (2, (4, 32, 128), 0.9, (512, 512, 2, 1)),          # 512 and 513: the other form for as many teams as fit, one wavefront an item
    (1, (4, 12, 684), 0.97, (513, 513, 1, 1)),
    (5, (4, 40, 64), 0.9, (800, 800, 1, 1)),           # 800 and 801, lists made inside; from lists of kernels in front
    (3, (4, 12, 356), 0.9, (801, 801, 1, 1)),
    (2, (4, 40, 160), 0.97, (800, 800, 1, 1)),
    (1, (8, 32, 32), 0.0, (128, 128, 4, 2)),           # parts of teams
    (2, (4, 32, 136), 0.2, (544, 544, 1, 3)),          # parts of one wavefront
    (1, (7, 31, 30), 0.0, (128, 128, 4, 2)),           # ... of lists of halves
    (2, (3, 30, 134), 0.1, None),
])
def test_few_items_equal_many(heads, latent, sparsity, split, dtype):
    """The same heads, with the lists that the call made, among so many that every item has one wavefront of the other kernel.  Two orders of the
    same fp32 sums and two roundings of P: max-abs 1.6e-2 and mean-abs 1e-3 of outputs near 1, lse 2e-3."""
    from longcat_video_amd import _capi
    from longcat_video_amd.block_sparse_attention import bsa_interface as bi
    S = math.prod(latent)
    g = torch.Generator(device="cuda").manual_seed(51)
    q, k, v = (torch.randn(1, heads, S, 128, generator=g, device="cuda").to(dtype) for _ in range(3))
    if split is not None:
        how = (ctypes.c_int32 * 4)()
        _capi.check(_capi.load().bsa_fwd_3d_last_round(bi._plan_of(1, heads, 128, bi._code(q), latent, latent, CHUNK, CHUNK, sparsity, None).prm, how))
        assert tuple(how) == split
    o, walk, lens, lse = bi._bsa_3d(q, k, v, latent, latent, sparsity, CHUNK, CHUNK, for_backward=True)
    many = -(-1100 // (heads * math.prod(-(-n // 4) for n in latent)))
    rep = lambda x: x.repeat(1, many, *([1] * (x.dim() - 2)))      # noqa: E731
    want, want_lse = bi.ThwAttention(rep(k), rep(v), latent, latent, CHUNK, CHUNK)(rep(q), rep(walk), rep(lens), return_lse=True)
    d = (o.float() - want[:, :heads].float()).abs()
    assert d.max() <= 1.6e-2 and d.mean() <= 1e-3, (float(d.max()), float(d.mean()))
    assert (lse - want_lse[:, :heads]).abs().max() <= 2e-3
    assert torch.equal(bi.flash_attn_bsa_3d(q, k, v, latent, latent, sparsity=sparsity, chunk_3d_shape_q=CHUNK, chunk_3d_shape_k=CHUNK), o)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_maxima_that_rise(dtype):
    """Keys that grow along the walk: the running maximum is raised again and again, in one wavefront an item, teams and parts."""
    from longcat_video_amd.block_sparse_attention import bsa_interface as bi
    latent = (8, 32, 32)
    S = math.prod(latent)
    g = torch.Generator(device="cuda").manual_seed(52)
    for heads in (1, 3, 5, 6):                  # teams of four in parts, of two, one wavefront, one wavefront
        q, k, v = (torch.randn(1, heads, S, 128, generator=g, device="cuda") for _ in range(3))
        k = k * torch.linspace(0.2, 6, S, device="cuda")[:, None]
        q, k, v = (x.to(dtype) for x in (q, k, v))
        o, walk, lens, lse = bi._bsa_3d(q, k, v, latent, latent, 0.0, CHUNK, CHUNK, for_backward=True)
        i = torch.randint(0, S, (64,), generator=torch.Generator().manual_seed(heads)).cuda()
        s = q[0, :, i].double() @ k[0].double().transpose(1, 2).contiguous() * 128 ** -0.5
        want_lse = torch.logsumexp(s, -1)
        want = torch.softmax(s, -1) @ v[0].double()
        assert (lse[0, :, i] - want_lse).abs().max() <= 2e-3
        assert (o[0, :, i].double() - want).abs().max() <= 3e-2          # P to 2^-9, values to 4.5, half an ulp of an output to 4 (2^-7)
