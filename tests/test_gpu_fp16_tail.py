"""fp16 probabilities far below a row's largest: fp16 ends at 2^-24, so how many bits they keep is decided by the reference that
the exponents are taken from."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("items,drop", [(1280, 22.1), (1280, 18.0), (320, 22.1)])
def test_probabilities_keep_their_bits_below_the_largest(items, drop):
    """A first block of keys sets a row's largest logit (6, log2), all others lie `drop` below it, and the norms of q and k would
    allow logits 18.5 above it.  Values are 0 on the first block and 100 on the others, so the output is the others' share
    alone.  With a reference no higher than the largest logit a probability of 2^-drop is a multiple of 2^-24 and at most half
    of one off: 2^(drop - 25) of itself, the same for every key here (plus 2^-9 for the scores of fp16 inputs in fp32 and
    the rounding of the output).  items: more than one round of the attention kernel, and less."""
    from longcat_video_amd.block_sparse_attention import bsa_interface as bi
    log2_scale = 128 ** -0.5 * math.log2(math.e)
    nbk, nbq = 64, items // 5
    q = torch.zeros(1, 5, nbq * 64, 128)
    q[..., 0] = 8
    k = torch.zeros(1, 5, nbk * 64, 128)
    v = torch.full_like(k, 100.0)
    k[..., 0] = (6 - drop) / (8 * log2_scale)
    k[..., 2] = 18
    k[:, :, :64, 0], k[:, :, :64, 2], v[:, :, :64] = 6 / (8 * log2_scale), 23.2, 0
    q, k, v = (x.half() for x in (q, k, v))
    idx = torch.arange(nbk, dtype=torch.int32).expand(1, 5, nbq, nbk).contiguous()
    lens = torch.full((1, 5, nbq), nbk, dtype=torch.int32)
    o, _ = bi.attn_fwd_bsa_varlen(q.cuda(), k.cuda(), v.cuda(), 128 ** -0.5, idx.cuda(), lens.cuda(), 64, 64, kernel="fragment")
    want = torch.softmax(q[0, 0, :1].double() @ k[0, 0].double().T * 128 ** -0.5, -1) @ v[0, 0].double()
    assert 0 < float(want.min()) == float(want.max())
    off = (o.cpu().double() / float(want[0, 0]) - 1).abs().max()
    assert off <= 2 ** (drop - 25) + 2 ** -9, float(off)
