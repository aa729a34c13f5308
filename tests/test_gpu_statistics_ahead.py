"""Order statistics of samples of three million values and more, where the first pass keeps the values that the second one
needs: against a sorted copy, also where its guess from the first rows is wrong or there are too many of them."""
import pytest

torch = pytest.importorskip("torch")

if torch.cuda.is_available():
    import f2cgt_amd

pytestmark = pytest.mark.gpu


def _table(kind, n, d, g):
    x = torch.randn((n, d), generator=g, device="cuda")
    if kind == "growing":                 # the first rows of a workgroup say little about its last
        x *= torch.logspace(-6, 6, n, device="cuda")[:, None]
    elif kind == "columns":
        x *= torch.exp(3 * torch.randn((1, d), generator=g, device="cuda"))
    elif kind == "few":                   # all of them share a handful of digits
        x = x.mul_(2).round_()
    elif kind == "special":
        x[::97] = float("inf")
        x[1::97] = 0.0
        x[2::97, ::3] = 1e-40
    return x


@pytest.mark.parametrize("kind", ["normal", "growing", "columns", "few", "special"])
# columns of four, two and one at a time; a narrow last slice; more column groups than threads; sizes about the line
@pytest.mark.parametrize("n,d,slice_", [(30001, 100, 104), (40000, 150, 64), (46155, 65, 65), (46153, 65, 65), (375000, 8, 8),
                                        (3000, 1030, 1030), (1500, 4100, 4100), (3000007, 1, 1)])
def test_ranks_and_sum(kind, n, d, slice_):
    g = torch.Generator(device="cuda")
    g.manual_seed(n + d)
    x = _table(kind, n + 30, d, g)
    rows = torch.arange(n, device="cuda") if kind == "growing" else torch.randint(-n, n + 30, (n,), generator=g, device="cuda")
    count = (d + slice_ - 1) // slice_
    for places in (lambda t: [t // 200, t // 200 + 1, t * 199 // 200, t * 199 // 200 + 1], lambda t: [0, t // 2, t // 3, t - 1],
                   lambda t: [t - 1, t // 100, 0, t // 50]):
        ranks = [r for i in (0, count - 1) for r in places(n * min(slice_, d - i * slice_))]
        got = f2cgt_amd.load().abs_order_stats(x, rows, slice_, ranks).cpu()
        sample = x[rows].abs()
        for i in range(count):
            part = sample[:, i * slice_:(i + 1) * slice_].reshape(-1)
            want = part.sort().values[torch.tensor(ranks[4:] if i == count - 1 else ranks[:4], device="cuda")]
            assert torch.equal(got[i, :4].float(), want.cpu()), (i, ranks)
            assert got[i, 5] == 0.0
            total = float(part.sum(dtype=torch.float64))
            # fp64 sums of non-negative values in any order: (number of terms) roundings of the total at most
            assert got[i, 4] == total if total == float("inf") else abs(float(got[i, 4]) - total) <= part.numel() * 2.0 ** -52 * total


def test_a_nan_and_a_bad_row_are_reported():
    x = torch.ones((40000, 100), device="cuda")
    x[39999, 99] = float("nan")
    lib = f2cgt_amd.load()
    ranks = [0, 1, 2, 3999999] * 2
    assert float(lib.abs_order_stats(x, None, 104, ranks)[0, 5]) == 1.0
    rows = torch.arange(40000, device="cuda")
    rows[39999] = 40000
    assert float(lib.abs_order_stats(x, rows, 104, ranks)[0, 5]) == 3.0      # (the clamped row is the one with the NaN)
