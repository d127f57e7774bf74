"""Selection on rows longer than the LDS schedule takes (the sampled schedule), where the threshold
lies among infinities, NaN, zeros of both signs or the lowest value, and at the sizes around its
16-key chunks: exactly the host routine's indices and mask."""
import pytest
import torch

from flash_evict import select_tokens

from _helpers import seeded_randn

pytestmark = pytest.mark.gpu

INF, NAN = float("inf"), float("nan")


@pytest.mark.parametrize("n", [16385, 16400, 33001, 131072])
@pytest.mark.parametrize("what", ["normal", "inf_many", "inf_few", "nan_many", "nan_few", "nan_and_inf", "minus_inf", "zeros"])
def test_sampled_schedule_matches_host(n, what):
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
    dev = x.cuda()
    for budget, recent, pool in ((n // 10, 0, 1), (64, 32, 1), (n // 2, 64, 1), (n - 5, 1, 1), (n // 20, 7, 5)):
        if pool > 1 and what not in ("normal", "zeros"):
            continue                              # pooled NaN and infinities: another input again
        idx, keep = select_tokens(dev, budget, recent=recent, pool_kernel=pool)
        hidx, hkeep = select_tokens(x, budget, recent=recent, pool_kernel=pool)
        assert torch.equal(idx.cpu(), hidx) and torch.equal(keep.cpu(), hkeep), (n, what, budget, recent, pool)
