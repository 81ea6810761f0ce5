"""The forward's left factor at the edges of its launch shapes: block rows on both sides of every 32-row query tile (one
wave up to a team of four, and a second grid slice past 128 rows), and columns whose rows two or four waves share."""
import pytest
import torch

import self_forcing_amd as sfa
from gpu_util import assert_close_16bit, randn
from oracle import monarch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _check(H, D, h, w, fq, fk, dtype, seed):
    q, k, v = (randn((1, f * h * w, H, D), seed + i, dtype) for i, f in enumerate((fq, fk, fk)))
    out = sfa.monarch_attn.monarch_attn(q.to(DEV), k.to(DEV), v.to(DEV), 1, 1, 1, h, w)
    ref = monarch.monarch_attn(q, k, v, 1, 1, 1, h, w, dtype=torch.float32)
    assert_close_16bit(out, ref, dtype)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("b1", [1, 31, 32, 33, 64, 65, 96, 97, 128, 129, 250])
def test_block_rows_around_query_tiles(b1, D):
    _check(2, D, b1, 3, 1, 2, torch.bfloat16, 900 + b1)


# (block rows, key frames): 1, 2, 4, 5, 8 and 13 chunks of 32 rows; five columns keep the chip empty, so that the rows are shared
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b1,fk", [(5, 4), (11, 4), (32, 4), (30, 5), (31, 8), (32, 8), (9, 45)])
@pytest.mark.parametrize("D", [64, 128])
def test_rows_shared_by_waves(b1, fk, D, dtype):
    _check(1, D, b1, 5, 1, fk, dtype, 950 + b1 + fk)
