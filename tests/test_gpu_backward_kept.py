"""dQ from the dS that the dK / dV kernel keeps, against dQ from scratch."""
import ctypes
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def run(q, k, v, do, idx, lens, stride, chunk_q, chunk_k):
    """The same lists in rows of `stride` entries (the workspace, and with it what is kept, is planned for full rows)."""
    from longcat_video_amd.block_sparse_attention import bsa_interface as bi
    wide = torch.zeros(*idx.shape[:-1], stride, dtype=torch.int32, device="cuda")
    wide[..., :idx.shape[-1]] = idx
    sm = 1 / math.sqrt(128)
    o, lse = bi.attn_fwd_bsa_varlen(q, k, v, sm, wide, lens, chunk_q, chunk_k)
    grads = [torch.full_like(t, float("nan")) for t in (q, k, v)]
    bi.attn_bwd_bsa_varlen(do, q, k, v, o, *grads, sm, lse, wide, lens, chunk_q, chunk_k)
    return grads


def case(heads, nbq, nbk, width, chunk_q, chunk_k, dtype, seed=41):
    g = torch.Generator(device="cuda").manual_seed(seed)
    new = lambda n: torch.randn(1, heads, n, 128, generator=g, device="cuda").to(dtype)      # noqa: E731
    q, do, k, v = new(nbq * chunk_q), new(nbq * chunk_q), new(nbk * chunk_k), new(nbk * chunk_k)
    idx = torch.rand(1, heads, nbq, nbk, generator=g, device="cuda").argsort(-1)[..., :width].int()
    lens = torch.randint(0, width + 1, (1, heads, nbq), generator=g, device="cuda").int()
    return q, k, v, do, idx, lens


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("chunk_q,chunk_k,nbq,nbk,wide", [(64, 64, 600, 900, 900), (128, 64, 300, 900, 900), (64, 128, 600, 450, 450), (192, 128, 200, 450, 450)])
def test_kept_ds_against_dq_from_scratch(dtype, chunk_q, chunk_k, nbq, nbk, wide):
    """Rows of full length need more than is kept (8 GB), short ones do not.
    dK and dV come from the same kernel: the same bits.  The two dQ start dP from 0 or from -delta, an fp32 rounding, so a dS
    may round the other way: an ulp of dS (2^-8, 2^-11) of one of up to 9 x 64 terms; a row's 2-norm stays within that."""
    q, k, v, do, idx, lens = case(3, nbq, nbk, 9, chunk_q, chunk_k, dtype)
    dq0, dk0, dv0 = run(q, k, v, do, idx, lens, 9, chunk_q, chunk_k)
    dq1, dk1, dv1 = run(q, k, v, do, idx, lens, wide, chunk_q, chunk_k)
    assert torch.equal(dk0, dk1) and torch.equal(dv0, dv1)
    ulp = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    assert torch.isfinite(dq0.float()).all()
    assert (dq0.float() - dq1.float()).norm() <= ulp * dq1.float().norm()



@pytest.mark.parametrize("grid,chunk", [((9, 17, 30), (4, 4, 4)), ((8, 8, 8), (4, 4, 8))])
def test_without_room_for_ds(grid, chunk, monkeypatch):
    """A workspace of the least size leaves dS out; tolerance as above, two ulps since both sides round dQ itself too."""
    from longcat_video_amd.block_sparse_attention import bsa_interface as bi
    g = torch.Generator(device="cuda").manual_seed(43)
    n = grid[0] * grid[1] * grid[2]
    q, k, v = (torch.randn(1, 2, n, 128, generator=g, device="cuda").half().requires_grad_() for _ in range(3))
    do = torch.randn(1, 2, n, 128, generator=g, device="cuda").half()
    args = dict(sparsity=0.5, chunk_3d_shape_q=list(chunk), chunk_3d_shape_k=list(chunk))

    def grads():
        return torch.autograd.grad(bi.flash_attn_bsa_3d(q, k, v, grid, grid, **args), (q, k, v), do)
    dq1, dk1, dv1 = grads()
    sizes = []

    def least_only(nbytes, least, device):
        sizes.append((nbytes, least))
        return torch.empty(least, dtype=torch.uint8, device=device)
    monkeypatch.setattr(bi, "_backward_workspace", least_only)
    dq0, dk0, dv0 = grads()
    assert sizes[0][1] < sizes[0][0]
    assert torch.equal(dk0, dk1) and torch.equal(dv0, dv1)
    assert (dq0.float() - dq1.float()).norm() <= 2 * 2.0 ** -11 * dq1.float().norm()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_lists_of_any_length_run_in_one_launch(dtype, monkeypatch):
    """2 304 query tiles and lists of 1 to 192 of 192 blocks, dQ from scratch: as wide as the blocks (one launch) and cut to the
    longest list (rounds), bit for bit the same."""
    from longcat_video_amd.block_sparse_attention import bsa_interface as bi
    lq, chunk, H = (12, 32, 32), (4, 4, 4), 12
    S = lq[0] * lq[1] * lq[2]
    g = torch.Generator("cuda").manual_seed(14)
    q, k, v, do = (torch.randn(1, H, S, 128, generator=g, device="cuda").to(dtype) for _ in range(4))
    lens = torch.randint(1, 40, (1, H, 192), generator=g, device="cuda", dtype=torch.int32)
    lens[..., ::37] = 150
    walk = torch.rand(1, H, 192, 192, generator=g, device="cuda").argsort(dim=-1).int()
    walk[..., :150] = walk[..., :150].sort(dim=-1).values
    o, lse = bi.ThwAttention(k, v, lq, lq, chunk, chunk)(q, walk, lens, return_lse=True)
    monkeypatch.setattr(bi, "_backward_workspace", lambda need, least, device: torch.empty(least, dtype=torch.uint8, device=device))
    wide, cut = (bi._bsa_3d_backward(do, q, k, v, o, lse, w, lens, lq, lq, chunk, chunk, 128 ** -0.5) for w in (walk, walk[..., :150].contiguous()))
    for a, b in zip(wide, cut):
        assert torch.isfinite(a.float()).all() and torch.equal(a, b)


def launches(f):
    """Nodes of the graph that a capture of f gives: its kernel launches."""
    f()                                              # set-up of the device, outside the capture
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        f()
    hip = next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64.so" in line)
    n = ctypes.c_size_t(0)
    count = ctypes.CDLL(hip).hipGraphGetNodes
    count.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.POINTER(ctypes.c_size_t)]
    assert count(graph.raw_cuda_graph(), None, ctypes.byref(n)) == 0
    return n.value


def test_launches_follow_the_rule_not_the_width(monkeypatch):
    """2 560 query tiles and every block kept, dS kept: rounds (two launches of dQ) for the top-k rule, whose lists are equal, one
    launch for the CDF rule, whose lists may be as wide; the same bits."""
    from longcat_video_amd.block_sparse_attention import bsa_interface as bi
    lq, chunk, H = (8, 16, 16), (4, 4, 4), 80
    S = lq[0] * lq[1] * lq[2]
    g = torch.Generator("cuda").manual_seed(16)
    q, k, v = (torch.randn(1, H, S, 128, generator=g, device="cuda").bfloat16().requires_grad_() for _ in range(3))
    do = torch.randn(1, H, S, 128, generator=g, device="cuda").bfloat16()
    calls, backward = [], bi._bsa_3d_backward
    monkeypatch.setattr(bi, "_bsa_3d_backward", lambda *a: calls.append(a) or backward(*a))
    grads = [torch.autograd.grad(bi.flash_attn_bsa_3d(q, k, v, lq, lq, chunk_3d_shape_q=chunk, chunk_3d_shape_k=chunk, **rule), (q, k, v), do)
             for rule in (dict(sparsity=0.0), dict(sparsity=0.0, cdf_threshold=0.5))]
    with torch.no_grad():
        counts = [launches(lambda: backward(*a)) for a in calls]      # noqa: B023
    assert counts[0] == counts[1] + 1, counts
    assert all(torch.isfinite(a.float()).all() and torch.equal(a, b) for a, b in zip(*grads))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_kept_ds_in_rounds_and_in_one_launch(dtype):
    """2 304 query tiles and lists of 1 to 150 of 192 blocks, dS kept: declared unequal (one launch) and not (rounds), as wide as the
    blocks and cut to the longest list, bit for bit the same."""
    from longcat_video_amd.block_sparse_attention import bsa_interface as bi
    lq, chunk, H = (12, 32, 32), (4, 4, 4), 12
    S = lq[0] * lq[1] * lq[2]
    g = torch.Generator("cuda").manual_seed(17)
    q, k, v, do = (torch.randn(1, H, S, 128, generator=g, device="cuda").to(dtype) for _ in range(4))
    lens = torch.randint(1, 40, (1, H, 192), generator=g, device="cuda", dtype=torch.int32)
    lens[..., ::37] = 150
    walk = torch.rand(1, H, 192, 192, generator=g, device="cuda").argsort(dim=-1).int()
    walk[..., :150] = walk[..., :150].sort(dim=-1).values
    o, lse = bi.ThwAttention(k, v, lq, lq, chunk, chunk)(q, walk, lens, return_lse=True)
    runs = [bi._bsa_3d_backward(do, q, k, v, o, lse, w, lens, lq, lq, chunk, chunk, 128 ** -0.5, unequal)
            for w in (walk, walk[..., :150].contiguous()) for unequal in (False, True)]
    for run_ in runs[1:]:
        assert all(torch.isfinite(a.float()).all() and torch.equal(a, b) for a, b in zip(run_, runs[0]))
