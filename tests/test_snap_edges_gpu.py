"""fe_snap_scores at keys with an infinite channel, beside padding rows (heads x window not a
multiple of the 32-row tile), at key blocks without one comparable logit (NaN), and with
probabilities in FP32's subnormal range."""
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


@pytest.mark.parametrize("hq,hk,n,d,w", [(4, 2, 700, 64, 32), (8, 1, 5000, 128, 20), (2, 1, 900, 256, 16),
                                         (16, 1, 1500, 64, 300)])
def test_subnormal_probabilities_are_kept(hq, hk, n, d, w):
    """Logits 0 for the first key and -75 to -99.75 for the others: probabilities of 2^-108 to 2^-144,
    two thirds of them below the smallest normal float. Bound: 2^-15 relative (the exponent's product
    by log2 e, up to 144, is rounded to 2^-17, its factor to 2^-25; v_exp_f32 and the reciprocal are
    far below that), one unit of 2^-149 for each row's two roundings and one for the mean."""
    print(f"snap_scores subnormals hq={hq} hk={hk} n={n} d={d} w={w}", flush=True)
    steps = 75 + 0.25 * (torch.arange(n) % 100).float()
    steps[0] = 0
    q = torch.zeros((1, hq, n, d), dtype=torch.float16)
    k = torch.zeros((1, hk, n, d), dtype=torch.float16)
    q[..., 0] = 8.0                                               # products by 8 are exact
    k[..., 0] = -(steps * d ** 0.5 / 8).to(torch.float16)
    got = snap_scores(q.cuda(), k.cuda(), w)
    torch.cuda.synchronize()
    logits = 8.0 * k[0, 0, :, 0].double() * d ** -0.5
    visible = torch.arange(n)[None, :] <= torch.arange(n - w, n)[:, None]
    p = torch.exp(logits)[None, :] * visible
    ref = (p / p.sum(1, keepdim=True)).sum(0)
    bound = 2.0 ** -15 * ref + (w + 1) * 2.0 ** -149
    err = (got.cpu().double() - ref).abs()
    assert (err <= bound).all(), float((err / bound).max())
    assert (got[..., :n - w] > 0).all()
