"""Gradients stored over the inputs."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def _backward(do, q, k, v, o, lse, walk, lens, lq, lk, chunk, dq, dk, dv, least=False):
    from longcat_video_amd import _capi
    from longcat_video_amd.block_sparse_attention import bsa_interface as bi
    B, H, _, D = q.shape
    prm, need, low = bi._plan_3d_backward(B, H, D, bi._code(q), *lq, *lk, *chunk, *chunk, 128 ** -0.5, walk.shape[3])
    ws = torch.empty(low if least else need, dtype=torch.uint8, device="cuda")
    at = lambda t: (bi._ptr(t), bi._st(t))      # noqa: E731
    _capi.check(_capi.load().bsa_bwd_3d(prm, *at(q), *at(k), *at(v), *at(o), *at(do), bi._ptr(lse), bi._ptr(walk), bi._ptr(lens),
                                        walk.shape[3], *at(dq), *at(dk), *at(dv), bi._ptr(ws), ws.numel(), bi._stream(q)), "bsa_bwd_3d")


@pytest.mark.parametrize("least", [False, True])
@pytest.mark.parametrize("where", ["own rows", "k and v exchanged", "dq over k", "dq over v", "other layout"])
@pytest.mark.parametrize("grid,chunk", [((8, 8, 16), (4, 4, 4)), ((5, 9, 13), (4, 4, 4))])
def test_gradients_over_the_inputs(grid, chunk, where, least):
    """The dK / dV kernel reads k and v where the caller has them.  dk and dv over their own rows, and gradients anywhere else over
    k or v, where the rows come from a copy: the bits of gradients in memory of their own (with dS kept on both sides or on neither;
    dQ alone is summed from other products where it is)."""
    from longcat_video_amd.block_sparse_attention import bsa_interface as bi
    S, H = math.prod(grid), 3
    g = torch.Generator(device="cuda").manual_seed(61)
    q, k, v, do = (torch.randn(1, H, S, 128, generator=g, device="cuda").bfloat16() for _ in range(4))
    o, walk, lens, lse = bi._bsa_3d(q, k, v, grid, grid, 0.5, chunk, chunk, for_backward=True)
    copies = where not in ("own rows", "k and v exchanged")
    want = [torch.empty_like(q) for _ in range(3)]
    _backward(do, q, k, v, o, lse, walk, lens, grid, grid, chunk, *want, least=least or copies)
    dq, dk, dv = (torch.empty_like(q) for _ in range(3))
    if where == "own rows":
        dk, dv = k, v
    elif where == "k and v exchanged":
        dk, dv = v, k
    elif where == "dq over k":
        dq = k
    elif where == "dq over v":
        dq = v
    else:                                        # [B, H, S, D] over the memory of a [B, S, H, D] view
        k, v = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in (k, v))
        dk, dv = (t.transpose(1, 2).view(1, H, S, 128) for t in (k, v))
    _backward(do, q, k, v, o, lse, walk, lens, grid, grid, chunk, dq, dk, dv, least=least)
    for a, b in zip((dq, dk, dv), want):
        assert torch.isfinite(a.float()).all() and torch.equal(a, b)


def test_blocked_gradients_over_the_keys():
    """The same for the blocked-order entry point: dq over k."""
    from longcat_video_amd.block_sparse_attention import bsa_interface as bi
    H, S = 2, 1024
    g = torch.Generator(device="cuda").manual_seed(62)
    q, k, v, do = (torch.randn(1, H, S, 128, generator=g, device="cuda").bfloat16() for _ in range(4))
    idx = torch.rand(1, H, S // 64, S // 64, generator=g, device="cuda").argsort(dim=-1)[..., :5].sort(dim=-1).values.int().contiguous()
    lens = torch.full((1, H, S // 64), 5, device="cuda", dtype=torch.int32)
    o, lse = bi.ThwAttention(k, v, (4, 4, 64), (4, 4, 64), (4, 4, 4), (4, 4, 4))(q, idx, lens, return_lse=True)
    outs = []
    for over in (False, True):
        kk = k.clone()
        dq, dk, dv = (torch.empty_like(q) for _ in range(3))
        if over:
            dq = kk
        bi.attn_bwd_bsa_varlen(do, q, kk, v, o, dq, dk, dv, 128 ** -0.5, lse, idx, lens, 64, 64, None, None)
        outs.append((dq, dk, dv))
    assert torch.equal(outs[0][1], outs[1][1]) and torch.equal(outs[0][2], outs[1][2])
    assert (outs[0][0].float() - outs[1][0].float()).norm() <= 2 * 2.0 ** -8 * outs[1][0].float().norm()
