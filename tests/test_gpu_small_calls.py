"""Kernels that small calls run: the fp32 attention kernel in both of its splits, and the gating in one launch."""
import math

import pytest
import torch

from oracle import bsa_oracle as O
from conftest import seeded_qkv

pytestmark = pytest.mark.gpu


def I():
    from longcat_video_amd.block_sparse_attention import bsa_interface
    return bsa_interface


@pytest.mark.parametrize("latent,chunk,heads,sparsity", [
    ((4, 8, 8), (4, 4, 4), 1, 0.75),        # one key block per row
    ((5, 9, 13), (4, 4, 4), 2, 0.5),        # ragged in every axis: whole key groups of padding
    ((3, 6, 12), (4, 4, 8), 3, 0.5),        # 128-slot chunks
    ((8, 32, 32), (4, 4, 4), 8, 0.875),     # 4 096 units of 16 rows: the last size of the split walk
    ((8, 32, 36), (4, 4, 4), 8, 0.9375),    # beyond it
])
def test_fp32_operator_against_the_oracle(latent, chunk, heads, sparsity):
    """fp32 products and sums in another order than the oracle's: 2e-5, the bound of the other fp32 tests."""
    S = math.prod(latent)
    q, k, v = seeded_qkv(71, 1, heads, S, S, 128, torch.float32)
    dev = [x.cuda() for x in (q, k, v)]
    o, idx, lens, score = I()._bsa_3d(*dev, latent, latent, sparsity, chunk, chunk, True)
    assert torch.equal(I().flash_attn_bsa_3d(*dev, latent, latent, sparsity=sparsity, chunk_3d_shape_q=chunk, chunk_3d_shape_k=chunk), o)
    bs = math.prod(chunk)
    kvalid = torch.from_numpy(O.slot_validity(latent, chunk))
    heads_checked = [0, heads - 1] if heads > 3 else list(range(heads))
    sub = lambda x: x[:, heads_checked]      # noqa: E731
    qp, kp, vp = (O.rearrange_thw_to_3d_block(sub(x), latent, chunk) for x in (q, k, v))
    mask = O.block_mask_from_indices(sub(idx).cpu().long(), sub(lens).cpu(), score.shape[-1])
    want, _ = O.masked_dense_attention(qp, kp, vp, mask, bs, bs, 1 / math.sqrt(128), key_valid=kvalid)
    want = O.rearrange_3d_block_to_thw(want, latent, chunk)
    assert (sub(o).cpu() - want).abs().max() <= 2e-5


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("latent,heads,sparsity", [
    ((4, 4, 8), 1, 0.5),           # two blocks, one kept
    ((4, 12, 44), 3, 0.5),         # 33 blocks: a second row group and a second column tile of one
    ((8, 32, 32), 2, 0.875),       # 128
    ((8, 34, 60), 2, 0.9),         # 270: not a multiple of 8
    ((16, 32, 64), 1, 0.75),       # 512: the widest, lists of 128
    ((16, 32, 68), 1, 0.75),       # 544: the separate kernels
])
def test_one_launch_gating_equals_the_separate_kernels(dtype, latent, heads, sparsity):
    """A call that asks for the selection runs score, top-k and visiting order one by one; the others gate in one launch
    where it is built.  The same lists in the same order give the same bits."""
    chunk, S = (4, 4, 4), math.prod(latent)
    q, k, v = (x.cuda() for x in seeded_qkv(72, 1, heads, S, S, 128, dtype))
    o = I()._bsa_3d(q, k, v, latent, latent, sparsity, chunk, chunk, True)[0]
    assert torch.equal(I().flash_attn_bsa_3d(q, k, v, latent, latent, sparsity=sparsity, chunk_3d_shape_q=chunk, chunk_3d_shape_k=chunk), o)


def test_a_rule_below_zero_is_none():
    """Called directly or through the custom op (a function mode sees the op go by), the arguments mean the same."""
    from longcat_video_amd.block_sparse_attention import bsa_interface as bi
    g = torch.Generator(device="cuda").manual_seed(3)
    grid, chunk = (4, 8, 16), [4, 4, 4]
    q, k, v = (torch.randn(1, 2, 512, 128, generator=g, device="cuda").bfloat16() for _ in range(3))
    kw = dict(chunk_3d_shape_q=chunk, chunk_3d_shape_k=chunk)
    seen = []

    class Mode(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))
    for rule in (dict(sparsity=0.5, cdf_threshold=-1.0), dict(sparsity=-0.5, cdf_threshold=0.5), dict(sparsity=0.5, cdf_threshold=0.0)):
        direct = bi.flash_attn_bsa_3d(q, k, v, grid, grid, **rule, **kw)
        with Mode():
            through = bi.flash_attn_bsa_3d(q, k, v, grid, grid, **rule, **kw)
        assert torch.equal(direct, through)
    assert any("bsa" in s for s in seen)
    want = bi.flash_attn_bsa_3d(q, k, v, grid, grid, sparsity=0.5, **kw)
    assert torch.equal(want, bi.flash_attn_bsa_3d(q, k, v, grid, grid, sparsity=0.5, cdf_threshold=-1.0, **kw))
    shape = [torch.tensor(x) for x in grid]      # sizes that are changed in place are not remembered
    assert torch.equal(want, bi.flash_attn_bsa_3d(q, k, v, shape, shape, sparsity=0.5, **kw))


def test_threads_with_different_lds_sizes():
    """Lists of 256 and of 496 blocks (84 and 130 KB of LDS for the one-launch gating), each from a host thread and on a
    stream of its own, at the same time: what each gives alone."""
    import threading
    latent, chunk = (16, 32, 64), (4, 4, 4)
    S, alone, got = math.prod(latent), {}, {0.5: [], 0.03125: []}
    q, k, v = (x.cuda() for x in seeded_qkv(73, 1, 1, S, S, 128, torch.bfloat16))
    call = lambda rule: I().flash_attn_bsa_3d(q, k, v, latent, latent, sparsity=rule, chunk_3d_shape_q=chunk, chunk_3d_shape_k=chunk)      # noqa: E731
    for rule in got:
        alone[rule] = call(rule)
    torch.cuda.synchronize()

    def work(rule):
        with torch.cuda.stream(torch.cuda.Stream()):
            got[rule] += [call(rule) for _ in range(20)]
            torch.cuda.current_stream().synchronize()
    threads = [threading.Thread(target=work, args=(rule,)) for rule in got]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for rule in got:
        assert len(got[rule]) == 20 and all(torch.equal(o, alone[rule]) for o in got[rule])


def test_values_that_are_not_in_memory():
    """A negated view and a zero tensor carry their sign, or all of their values, as a mark that the dispatcher resolves for
    operators that do not know of it; the direct call goes by the dispatcher and has to do the same."""
    g = torch.Generator(device="cuda").manual_seed(4)
    grid, rule = (4, 8, 16), dict(sparsity=0.5, chunk_3d_shape_q=[4, 4, 4], chunk_3d_shape_k=[4, 4, 4])
    q, k, v = (torch.randn(1, 2, 512, 128, generator=g, device="cuda").bfloat16() for _ in range(3))
    want = I().flash_attn_bsa_3d(-q, k, v, grid, grid, **rule)
    assert not torch.equal(want, I().flash_attn_bsa_3d(q, k, v, grid, grid, **rule))
    assert torch.equal(want, I().flash_attn_bsa_3d(torch._neg_view(q), k, v, grid, grid, **rule))
    nothing = torch._efficientzerotensor(v.shape, dtype=v.dtype, device="cuda")
    assert torch.equal(I().flash_attn_bsa_3d(q, k, nothing, grid, grid, **rule), torch.zeros_like(v))
