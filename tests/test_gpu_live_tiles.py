"""Query tiles without real rows left out of the attention kernel's work: ragged grids in chunks of several tiles."""
import numpy as np
import pytest
import torch

from conftest import seeded_qkv
from test_gpu_e2e import I, check_against_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("latent,chunk,heads", [
    ((5, 6, 13), (4, 4, 8), 2),        # one round; chunks with 40, 32 and 10 rows in their two tiles
    ((4, 9, 9), (4, 8, 8), 1),         # 256-slot chunks with 256, 32 and 4 rows
    ((4, 9, 17), (3, 8, 8), 2),        # 192 slots: 64 rows are one tile, 24 a part of one
    ((13, 30, 53), (4, 4, 8), 3),      # more than one round: items of two kinds of numbers in one launch
])
def test_ragged_chunks_of_several_tiles(latent, chunk, heads):
    S = int(np.prod(latent))
    q, k, v = seeded_qkv(31, 1, heads, S, S, 128, torch.bfloat16)
    o, idx, lens, score = I()._bsa_3d(q.cuda(), k.cuda(), v.cuda(), latent, latent, 0.5, chunk, chunk, True)
    nb = score.shape[-2]
    step = 1 if nb <= 16 else 13
    check_against_oracle(q, k, v, latent, latent, 0.5, o, idx, lens, score, list(range(0, nb, step)) + [nb - 1], chunk=chunk)
