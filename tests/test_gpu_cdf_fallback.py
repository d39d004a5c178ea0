"""Lists of unequal length with more work items than one round holds: the schedule that draws the items longest list first
runs the attention kernel without row maxima, and what that kernel leaves over has to be computed behind it as it is behind the
rounds."""
import pytest
import torch

pytestmark = pytest.mark.gpu
CHUNK, LATENT, HEADS = (4, 4, 4), (8, 32, 32), 9            # 1 152 work items: the rounds hold 1 024


def bi():
    from longcat_video_amd.block_sparse_attention import bsa_interface
    return bsa_interface


def inputs(dtype, size):
    """Nine chunks of ten point in one direction each (peaked pooled scores, short lists), the tenth has independent rows (flat
    scores, long lists), so the longest-first schedule wins.  Norms of 11 and 11 size: 8 in bf16 gives
    bounds on the logits beyond what the kernel without row maxima takes (fp16 always looks at the maxima)."""
    S = LATENT[0] * LATENT[1] * LATENT[2]
    g = torch.Generator().manual_seed(91)
    q, k, v = (torch.randn(1, HEADS, S, 128, generator=g) for _ in range(3))
    pos = torch.arange(S)
    chunk = ((pos // 1024) // 4) * 64 + (((pos // 32) % 32) // 4) * 8 + (pos % 32) // 4
    peaked = chunk % 10 != 0
    direction = torch.randn(1, HEADS, S // 64, 128, generator=g)[:, :, chunk]
    for x in (q, k):
        x[:, :, peaked] = size * direction[:, :, peaked] + 0.1 * x[:, :, peaked]
    return tuple(x.to(dtype).cuda() for x in (q, k, v))


def lists_of(q, k, v):
    _, idx, lens, _ = bi()._bsa_3d(q, k, v, LATENT, LATENT, None, CHUNK, CHUNK, True, cdf_threshold=0.5)
    assert int(lens.max()) > 4 * int(lens.min())
    asc = torch.where(idx < 0, torch.full_like(idx, 1 << 20), idx).sort(dim=-1).values
    asc = torch.where(asc == 1 << 20, torch.zeros_like(asc), asc)
    return bi().visit_order(asc.int(), lens, 128), lens      # the operator's visiting order


@pytest.mark.parametrize("dtype,size", [(torch.float16, 3.0), (torch.float16, 1.0), (torch.bfloat16, 8.0)])
def test_items_without_a_bound_are_computed(dtype, size):
    """Every row of o and lse, bit for bit what plain rounds give on the same lists, into a buffer full of NaN."""
    q, k, v = inputs(dtype, size)
    walk, lens = lists_of(q, k, v)
    rounds, lse = bi().ThwAttention(k, v, LATENT, LATENT, CHUNK, CHUNK)(q, walk, lens, return_lse=True)
    out = torch.full_like(q, float("nan"))
    bi()._bsa_3d(q, k, v, LATENT, LATENT, None, CHUNK, CHUNK, out=out, cdf_threshold=0.5)
    assert torch.equal(out, rounds)
    out = torch.full_like(q, float("nan"))
    either = bi().ThwAttention(k, v, LATENT, LATENT, CHUNK, CHUNK, unequal_lengths=True)
    _, lse2 = either(q, walk, lens, return_lse=True, out=out)
    assert torch.equal(out, rounds) and torch.equal(lse2, lse)


def test_gradients_of_items_without_a_bound():
    """The backward takes o and lse from the same call: the gradients of plain rounds, bit for bit."""
    q, k, v = inputs(torch.float16, 1.0)
    walk, lens = lists_of(q, k, v)
    o, lse = bi().ThwAttention(k, v, LATENT, LATENT, CHUNK, CHUNK)(q, walk, lens, return_lse=True)
    do = torch.randn(q.shape, generator=torch.Generator("cuda").manual_seed(92), device="cuda").half()
    want = bi()._bsa_3d_backward(do, q, k, v, o, lse, walk, lens, LATENT, LATENT, CHUNK, CHUNK, 128 ** -0.5)
    for x in (q, k, v):
        x.requires_grad_()
    got_o = bi().flash_attn_bsa_3d(q, k, v, LATENT, LATENT, sparsity=None, cdf_threshold=0.5, chunk_3d_shape_q=CHUNK, chunk_3d_shape_k=CHUNK)
    assert torch.equal(got_o, o)
    for got, ref in zip(torch.autograd.grad(got_o, (q, k, v), do), want):
        assert torch.isfinite(ref).all() and torch.equal(got, ref)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_an_infinite_key_reaches_the_output(dtype):
    """A head with an infinite key has no bound at all: its rows are computed, and those that see the key are not finite."""
    q, k, v = inputs(dtype, 1.0)
    k[0, 4, 777] = float("inf")
    walk, lens = lists_of(q, k, v)
    rounds = bi().ThwAttention(k, v, LATENT, LATENT, CHUNK, CHUNK)(q, walk, lens)
    out = torch.full_like(q, 7.0)
    bi()._bsa_3d(q, k, v, LATENT, LATENT, None, CHUNK, CHUNK, out=out, cdf_threshold=0.5)
    assert torch.equal(out.nan_to_num(nan=5.0), rounds.nan_to_num(nan=5.0))
    assert not torch.isfinite(out[0, 4]).all() and torch.isfinite(out[0, 3]).all()


@pytest.mark.parametrize("latent,heads,chunk,dtype", [
    ((13, 30, 53), 9, (4, 4, 8), torch.bfloat16),      # 3 339 of 4 032 query tiles hold rows: sections of 417 and 418 of them
    ((13, 30, 53), 9, (4, 4, 8), torch.float16),
    ((8, 33, 32), 15, (4, 4, 4), torch.bfloat16),      # 2 160 tiles: more items than the device runs at once, twice over
])
def test_queues_cover_ragged_grids(latent, heads, chunk, dtype):
    """Every row is computed once, whichever XCD's queue it is drawn from, on grids whose query tiles drop out or hold few rows.
    Bit for bit the rounds on the same lists."""
    T, H, W = latent
    S = T * H * W
    g = torch.Generator().manual_seed(93)
    q, k, v = (torch.randn(1, heads, S, 128, generator=g) for _ in range(3))
    pos = torch.arange(S)
    nh, nw = -(-H // chunk[1]), -(-W // chunk[2])
    block = ((pos // (H * W)) // chunk[0]) * nh * nw + (((pos // W) % H) // chunk[1]) * nw + (pos % W) // chunk[2]
    peaked = block % 10 != 0
    direction = torch.randn(1, heads, int(block.max()) + 1, 128, generator=g)[:, :, block]
    for x in (q, k):
        x[:, :, peaked] = 3 * direction[:, :, peaked] + 0.1 * x[:, :, peaked]
    q, k, v = (x.to(dtype).cuda() for x in (q, k, v))
    _, idx, lens, _ = bi()._bsa_3d(q, k, v, latent, latent, None, chunk, chunk, True, cdf_threshold=0.5)
    # what the choice on the device takes the queues for: long lists in every round of 1 024 items, and few of them
    tiles = -(-heads * lens.shape[-1] * chunk[2] // 4 // 1024)
    assert 1.4 * float(lens.float().sum()) * (chunk[2] // 4) / 1024 + int(lens.max()) < 0.9 * tiles * int(lens.max())
    nbk = int(block.max()) + 1
    asc = torch.where(idx < 0, torch.full_like(idx, 1 << 20), idx).sort(dim=-1).values
    walk = bi().visit_order(torch.where(asc == 1 << 20, torch.zeros_like(asc), asc).int(), lens, nbk)
    rounds = bi().ThwAttention(k, v, latent, latent, chunk, chunk)(q, walk, lens)
    out = torch.full_like(q, float("nan"))
    bi()._bsa_3d(q, k, v, latent, latent, None, chunk, chunk, out=out, cdf_threshold=0.5)
    assert torch.equal(out, rounds)
