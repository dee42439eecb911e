"""adana_order_stats_sampled (adana_amd/csrc/adana_order_sampled.h) where it can
go wrong, against np.sort: the sizes around the in-LDS sort, a tile and the bin
budgets, aligned and not, and values that crowd into few bins, repeat, sit far
outside the sample or make a tensor fall back to the radix select.  Selected
values are the tensor's own, so every comparison is exact."""
import numpy as np
import pytest
import torch

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a ROCm GPU")]

DEV = "cuda:0"

KINDS = {
    "cluster": lambda r, n: 0.4 + 0.0126 * r.standard_normal(n),
    "spread": lambda r, n: 10.0 ** (-3.0 * r.random(n)),
    "both signs": lambda r, n: r.standard_normal(n),
    "half zero": lambda r, n: np.where(r.random(n) < 0.5, 0.0, 0.4 + 0.01 * r.standard_normal(n)),
    "two repeated": lambda r, n: np.select([r.random(n) < 0.3, r.random(n) < 0.3], [0.0, 0.41], 0.4 + 0.01 * r.standard_normal(n)),
    "repeated NaN": lambda r, n: np.where(r.random(n) < 0.2, np.nan, 1.0 + 0.1 * r.standard_normal(n)),
    "constant": lambda r, n: np.full(n, 0.25),
    "few values (radix)": lambda r, n: r.integers(0, 40, n) / 8.0,
    "one narrow cluster (radix)": lambda r, n: 1.0 + 1e-6 * r.standard_normal(n),
    "far outliers": lambda r, n: np.where(np.arange(n) % max(n // 5, 1) == 1, -np.inf, 1.0 + 1e-2 * r.standard_normal(n)),
    "sorted": lambda r, n: np.sort(r.random(n)),
    "descending": lambda r, n: -np.sort(r.random(n)),
}
SIZES = (8191, 8192, 8193, 16384, 16387, 65537, (1 << 19) - 1, (1 << 19) + 5, (1 << 21) + 3)


def _check(xs, ranks):
    from adana_amd.tau_stats import order_values

    got = order_values(xs, ranks)
    for x, r, g in zip(xs, ranks, got):
        want = np.sort(x.cpu().numpy())[r]
        assert np.array_equal(g, want, equal_nan=True)


@pytest.mark.parametrize("n", SIZES)
def test_every_kind_at_the_edges(n):
    """Every kind of values in one batch, whole (16-byte aligned) and from the
    second value on (4 bytes off, one value less)."""
    from adana_amd.tau_stats import _rank_plan

    print(f"case: sampled order statistics, {n} values of {len(KINDS)} kinds", flush=True)
    rng = np.random.default_rng(n)
    xs = [torch.from_numpy(f(rng, n).astype(np.float32)).to(DEV) for f in KINDS.values()]
    xs += [x[1:] for x in xs]
    _check(xs, [_rank_plan(x.numel())[0] for x in xs])


@pytest.mark.parametrize("count", [1, 5, 1023, 1024, 1025])
def test_rank_counts(count):
    """Up to 1,024 ranks per tensor take the sampled path, more the radix
    select; given shuffled and repeated, and crowded into one bin."""
    rng = np.random.default_rng(count)
    n = 600_001
    print(f"case: sampled order statistics, {count} ranks", flush=True)
    x = torch.from_numpy((0.4 + 0.0126 * rng.standard_normal(n)).astype(np.float32)).to(DEV)
    spread = rng.permutation(rng.integers(0, n, count))
    crowded = np.minimum(300_000 + np.arange(count), n - 1)
    _check([x, x], [spread, crowded])


def test_large_bins():
    """A tensor whose bins hold more candidates than one workgroup's registers
    (the large-segment kernel), with outer bins of far more than its LDS sort
    takes: 48M values over 30 decades, smallest and largest ones crowded."""
    from adana_amd.tau_stats import _rank_plan

    n = 48_000_003
    print(f"case: sampled order statistics, {n} values", flush=True)
    g = torch.Generator(device=DEV)
    g.manual_seed(3)
    x = torch.pow(10.0, 30.0 * torch.rand(n, device=DEV, generator=g) - 20.0)
    x[::1500] *= 1e-12
    ranks = _rank_plan(n)[0]
    from adana_amd.tau_stats import order_values

    (got,) = order_values([x], [ranks])
    want = torch.sort(x)[0][torch.tensor(ranks, device=DEV)].cpu().numpy()
    assert np.array_equal(got, want)


@pytest.mark.parametrize("outliers", [0, 2000])
@pytest.mark.parametrize("width", [1, 3, 40, 300])
def test_clusters_of_few_keys(width, outliers):
    """Nearly all values on ``width`` neighbouring floats, the rest spread over
    many decades: too narrow for the bins, so left to the radix select (by the
    sample, or after the first read): the same values as np.sort's."""
    from adana_amd.tau_stats import order_values

    print("case: cluster", width, outliers, flush=True)
    rng = np.random.default_rng(width)
    n = 200_000
    x = (np.float32(0.25).view(np.int32) + rng.integers(0, width, n).astype(np.int32)).view(np.float32)
    at = rng.choice(n, outliers, replace=False)
    x[at] = (10.0 ** rng.uniform(-30, 0, outliers)).astype(np.float32)
    ranks = np.unique(np.concatenate([np.arange(0, n, 997), [0, n - 1]])).astype(np.int64)
    got = order_values([torch.from_numpy(x).to(DEV)], [ranks])[0]
    np.testing.assert_array_equal(np.asarray(got), np.sort(x)[ranks])
