"""bf16 linear layers with a residual: bf16(x w^T + bias + residual), by the engine's GEMM where it serves them, otherwise an fp32
product of the library and a pass that adds the rest."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def M():
    from longcat_video_amd.modules import attention
    return attention


def _integers(g, *shape):
    return torch.randint(-2, 3, shape, generator=g, device="cuda").bfloat16()


@pytest.mark.parametrize("with_bias", [True, False])
@pytest.mark.parametrize("rows,cols,k,in_place", [
    (1, 8, 64, False),
    (257, 384, 512, False),
    (300, 100, 60, False),            # columns that 16-byte pieces do not divide
    (33, 4100, 128, True),
    (3000, 4096, 64, True),           # by the engine's GEMM
    (3, 8388616, 8, False),           # the least workspace does not take all columns of a row
])
def test_sums_are_rounded_once(rows, cols, k, with_bias, in_place):
    """Small integers: every sum is exact in fp32, so the result is the exact one, rounded, whatever the workspace and the groups of
    rows that it makes."""
    g = torch.Generator(device="cuda").manual_seed(41)
    x, w, r = _integers(g, rows, k), _integers(g, cols, k), _integers(g, rows, cols) * 37
    b = _integers(g, cols) * 5 if with_bias else None
    want = x.float() @ w.float().t() + r.float()
    if with_bias:
        want += b.float()
    want = want.bfloat16()
    for workspace in (None, torch.empty(64 << 20, dtype=torch.uint8, device="cuda")):
        res = r.clone()
        got = M().linear_bf16(x, w, b, residual=res, workspace=workspace, out=res if in_place else None)
        assert torch.equal(got, want)


@pytest.mark.parametrize("in_place", [False, True])
@pytest.mark.parametrize("with_bias", [True, False])
@pytest.mark.parametrize("rows,cols,k", [
    (4500, 4096, 320),                # 288 tiles in two rounds of 256: 2 048 rows at a time, the last group of 404
    (3000, 4100, 64),                 # columns that the engine's GEMM does not take: 1 792 (of 2 046) and 1 208
])
def test_groups_of_rows_of_the_library_route(rows, cols, k, with_bias, in_place):
    from longcat_video_amd import _capi
    lib = _capi.load()
    g = torch.Generator(device="cuda").manual_seed(44)
    x, w, r = _integers(g, rows, k), _integers(g, cols, k), _integers(g, rows, cols) * 37
    b = _integers(g, cols) * 5 if with_bias else None
    want = x.float() @ w.float().t() + r.float()
    if with_bias:
        want += b.float()
    out = r.clone() if in_place else torch.empty_like(r)
    res = out if in_place else r
    p = lambda t: None if t is None else t.data_ptr()      # noqa: E731
    need = lib.bsa_linear_bf16_ld_workspace_bytes(p(x), k, p(w), k, p(b), p(res), p(out), cols, rows, cols, k)
    assert need > (64 << 20) + rows * cols * 4      # the library's: room for the whole product
    edge, room = 1 << 20, 64 << 20
    around = torch.full((room + 2 * edge,), 0x5a, dtype=torch.uint8, device="cuda")
    got = M().linear_bf16(x, w, b, residual=res, workspace=around[edge:edge + room], out=out)
    assert torch.equal(got, want.bfloat16())
    assert (around[:edge] == 0x5a).all() and (around[edge + room:] == 0x5a).all()


def test_strided_rows():
    """Row strides longer than the rows, of 16-byte pieces and not; nothing is written between the rows."""
    from longcat_video_amd import _capi
    lib = _capi.load()
    g = torch.Generator(device="cuda").manual_seed(42)
    ws = torch.empty(64 << 20, dtype=torch.uint8, device="cuda")
    for cols, pitch in ((64, 96), (64, 77), (50, 64)):
        x, w, b = _integers(g, 70, 48), _integers(g, cols, 48), _integers(g, cols)
        r, out = _integers(g, 70, pitch), torch.full((70, pitch), 7.0, dtype=torch.bfloat16, device="cuda")
        p = lambda t: t.data_ptr()      # noqa: E731
        _capi.check(lib.bsa_linear_bf16_ld(p(x), 48, p(w), 48, p(b), p(r), p(out), pitch, 70, cols, 48, p(ws), ws.numel(),
                                           torch.cuda.current_stream().cuda_stream), "linear")
        want = (x.float() @ w.float().t() + b.float() + r[:, :cols].float()).bfloat16()
        assert torch.equal(out[:, :cols], want) and (out[:, cols:] == 7).all()


def test_equal_calls_are_equal_at_720p_size():
    """The output projection of a 720p block, 2 000 times (by the engine's GEMM, which serves it).  With the residual added by the library's product (beta = 1) one call in 550 to
    830 came out with wrong rows."""
    g = torch.Generator(device="cuda").manual_seed(43)
    rows, dim = 86400, 4096
    x, r = (torch.randn(rows, dim, generator=g, device="cuda", dtype=torch.float32).bfloat16() for _ in range(2))
    w = (torch.randn(dim, dim, generator=g, device="cuda") * 0.02).bfloat16()
    b = torch.randn(dim, generator=g, device="cuda").bfloat16()
    out = torch.empty(rows, dim, dtype=torch.bfloat16, device="cuda")
    want = M().linear_bf16(x, w, b, residual=r, out=out).clone()
    for i in range(2000):
        assert torch.equal(M().linear_bf16(x, w, b, residual=r, out=out), want), i
