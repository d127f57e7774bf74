"""Selection on rows longer than the LDS schedule takes (the sampled schedule: more than 16384 keys
before the recent suffix), where the threshold lies among infinities, NaN, zeros of both signs or the
lowest value, at the sizes around its 16-key chunks, and on both sides of the most kept indices that
leave through LDS: exactly the host routine's indices and mask."""
import pytest
import torch

from flash_evict import select_tokens

from _helpers import seeded_randn

pytestmark = pytest.mark.gpu

INF, NAN = float("inf"), float("nan")


PAIRS = ((0.1, 0, 1), (64, 32, 1), (0.5, 64, 1), (-5, 1, 1), (0.05, 7, 5))   # past keys kept (share, number, all but), recent, pool


@pytest.mark.parametrize("past", [16385, 16399, 16400, 16401, 33001, 131072])
@pytest.mark.parametrize("what", ["normal", "inf_many", "inf_few", "nan_many", "nan_few", "nan_and_inf", "minus_inf", "zeros"])
def test_sampled_schedule_matches_host(past, what):
    n = past + 64
    x = seeded_randn((3, n), torch.float32, n + len(what), device="cpu")
    g = torch.Generator().manual_seed(n)
    pick = torch.rand((3, n), generator=g)
    if what == "inf_many":
        x[pick < 0.3] = INF
    elif what == "inf_few":
        x[pick < 0.004] = INF
    elif what == "nan_many":
        x[pick < 0.3] = NAN
    elif what == "nan_few":
        x[pick < 0.004] = NAN
    elif what == "nan_and_inf":
        x[pick < 0.05] = NAN
        x[(pick >= 0.05) & (pick < 0.15)] = INF
    elif what == "minus_inf":
        x[pick < 0.95] = -INF
    elif what == "zeros":
        x[pick < 0.5] = 0.0
        x[pick < 0.25] = -0.0
    for kept, recent, pool in PAIRS:
        if pool > 1 and what not in ("normal", "zeros"):
            continue                              # pooled NaN and infinities: another input again
        row = x[:, :past + recent].contiguous()
        kept = int(past * kept) if isinstance(kept, float) else kept if kept > 0 else past + kept
        _check(row, kept + recent, recent, pool, what)


def _check(row, budget, recent, pool, what):
    idx, keep = select_tokens(row.cuda(), budget, recent=recent, pool_kernel=pool)
    hidx, hkeep = select_tokens(row, budget, recent=recent, pool_kernel=pool)
    assert torch.equal(idx.cpu(), hidx) and torch.equal(keep.cpu(), hkeep), (tuple(row.shape), what, budget, recent, pool)


@pytest.mark.parametrize("past", [32773, 40000, 131072])
@pytest.mark.parametrize("kept", [24575, 24576, 24577])
@pytest.mark.parametrize("what", ["normal", "ties"])
def test_kept_indices_on_both_sides_of_the_staging_limit(past, kept, what):
    """Up to 24576 kept indices of the past leave through LDS, more are stored where they are found.
    "ties": nine values, so that the threshold lies among thousands of equal keys."""
    for recent in (0, 33):
        row = seeded_randn((2, past + recent), torch.float32, past + kept, device="cpu")
        if what == "ties":
            row = (2 * row).round().clamp(-4, 4)
        _check(row, kept + recent, recent, 1, what)
