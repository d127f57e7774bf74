"""fe_snap_scores over its block shapes: key groups per block (8 down to 1, by the key count),
64 or 32 keys per group, row parts, more than one chunk of row tiles per block, and windows of
more rows per group than a block keeps statistics of (the combine kernel), up to those whose partials
cover several key blocks. Against the oracle,
with the tolerance of test_snap_gpu (a logit near a rounding boundary may land one ulp of the
input type apart)."""
import pytest
import torch

from flash_evict.baselines import snap_scores
from oracle import snap as osnap

from test_snap_gpu import _check_scores, _qk

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,hq,hk,n,d,w,dtype,layout", [
    (1, 2, 1, 31, 128, 31, torch.bfloat16, "contiguous"),        # one group of 32 keys, every key masked somewhere
    (1, 8, 2, 8193, 128, 33, torch.bfloat16, "transposed"),      # 32-key groups, 8 row parts, a last block of one key
    (1, 4, 4, 8192, 64, 32, torch.float16, "contiguous"),        # 64-key groups, 4 row parts
    (2, 14, 2, 9000, 128, 128, torch.bfloat16, "transposed"),    # 28 row tiles: four chunks, 128-key blocks
    (4, 8, 8, 4100, 128, 40, torch.float16, "contiguous"),       # 512-key blocks, ragged
    (1, 8, 8, 16500, 256, 20, torch.bfloat16, "contiguous"),     # tile dim 256: four waves
    (1, 16, 1, 700, 64, 300, torch.bfloat16, "contiguous"),      # 4800 rows per group: combine kernel, three LDS loads
    (1, 16, 2, 400, 72, 256, torch.float16, "channel_stride2"),  # exactly 2048 rows, element loads
    (1, 32, 1, 1536, 64, 1536, torch.bfloat16, "contiguous"),    # 1536 row tiles: 2 key blocks per partial, row parts
    (1, 20, 1, 1999, 200, 1999, torch.float16, "transposed"),    # 2 of 63 key blocks per partial, rows ragged, four waves
    (1, 2, 1, 6001, 64, 6001, torch.bfloat16, "contiguous"),     # rows whose last position is before a block's keys
    (2, 64, 1, 1100, 32, 1100, torch.bfloat16, "transposed"),    # 3 key blocks per partial, 2 in the last
])
def test_snap_block_shapes_match_oracle(b, hq, hk, n, d, w, dtype, layout):
    print(f"snap_scores blocks b={b} hq={hq} hk={hk} n={n} d={d} w={w} {dtype} {layout}", flush=True)
    q, k = _qk(b, hq, hk, n, d, dtype, 4000 + n + d, layout)
    got = snap_scores(q, k, w)
    torch.cuda.synchronize()
    _check_scores(got, osnap.snap_scores(q.cpu(), k.cpu(), w), min(w, n))


@pytest.mark.parametrize("w", [32, 2100])
def test_rows_of_minus_infinity_contribute_nothing(w):
    """fp16 products below -65504 round to -inf; a row whose every logit is -inf has no softmax and
    adds nothing to any key (w = 2100: statistics from the combine kernel). The other head's rows
    are unchanged by it."""
    n, d = 2500, 128
    q, k = _qk(1, 2, 1, n, d, torch.float16, 77)
    k[...] = -k.abs() - 1
    q[:, 0] = 500.0
    got = snap_scores(q, k, w)
    alone = snap_scores(q[:, 1:].contiguous(), k, w)
    torch.cuda.synchronize()
    assert torch.isfinite(got).all()
    torch.testing.assert_close(got, alone / 2, rtol=1e-5, atol=0)
