"""fe_snap_scores at keys with an infinite channel, beside padding rows (heads x window not a
multiple of the 32-row tile), and at key blocks without one comparable logit (NaN)."""
import pytest
import torch

from flash_evict.baselines import snap_scores, snap_select
from oracle import snap as osnap

from test_snap_gpu import _check_scores, _qk

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,hq,hk,n,d,w,dtype,layout", [
    (1, 7, 1, 600, 128, 16, torch.bfloat16, "contiguous"),       # 112 rows: 16 of padding
    (2, 10, 2, 9000, 64, 20, torch.float16, "transposed"),       # 100 rows
    (1, 7, 1, 2000, 256, 9, torch.bfloat16, "contiguous"),       # 63 rows, four waves
    (1, 16, 2, 1500, 72, 3, torch.float16, "channel_stride2"),   # 24 rows, element loads
    (1, 16, 1, 2000, 64, 257, torch.bfloat16, "contiguous"),     # 4112 rows: statistics merged once
])
def test_padding_rows_add_nothing_to_a_key_with_an_infinite_channel(b, hq, hk, n, d, w, dtype, layout):
    """A key masked out by -inf in one channel (positive in every query) has probability 0 in every
    row; the padding rows' zero query times that infinity is NaN and must not reach the score."""
    print(f"snap_scores infinite channel b={b} hq={hq} hk={hk} n={n} d={d} w={w} {dtype} {layout}", flush=True)
    q, k = _qk(b, hq, hk, n, d, dtype, 9000 + n + d, layout)
    q[..., 5] = q[..., 5].abs() + 0.5
    masked = [3, 64, n // 2, n - w - 1]
    k[:, :, masked, 5] = float("-inf")
    got = snap_scores(q, k, w)
    torch.cuda.synchronize()
    assert torch.isfinite(got).all()
    assert (got[..., masked] == 0).all()
    _check_scores(got, osnap.snap_scores(q.cpu(), k.cpu(), w), w)
    _, keep = snap_select(got, n // 2, w, 1)
    assert not keep[..., masked].any()


@pytest.mark.parametrize("b,hq,hk,n,d,w,dtype,lo,hi", [
    (1, 8, 2, 3000, 128, 32, torch.bfloat16, 128, 1280),
    (2, 4, 2, 9000, 64, 128, torch.float16, 64, 2048),
    (1, 4, 1, 5000, 256, 40, torch.bfloat16, 4096, 4864),
    (1, 16, 1, 2000, 64, 300, torch.bfloat16, 192, 1024),        # statistics merged once
])
def test_key_blocks_of_nan_reach_every_score(b, hq, hk, n, d, w, dtype, lo, hi):
    """Keys lo .. hi-1 (multiples of 64) are NaN, so that some waves hold no other key: every row's
    softmax has NaN terms, and every score is NaN, as for a single such key."""
    print(f"snap_scores NaN blocks b={b} hq={hq} hk={hk} n={n} d={d} w={w} {dtype} {lo}:{hi}", flush=True)
    q, k = _qk(b, hq, hk, n, d, dtype, 9100 + n + d)
    k[:, :, lo:hi, 1] = float("nan")
    got = snap_scores(q, k, w)
    torch.cuda.synchronize()
    assert torch.isnan(osnap.snap_scores(q.cpu(), k.cpu(), w)).all()
    assert torch.isnan(got).all()
