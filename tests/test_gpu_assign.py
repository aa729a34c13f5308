"""Nearest-centre labels on the matrix cores (assign_kernel) against float64 distances of the original values: the labels
are the true first minimum, so they have to be equal wherever the two smallest float64 distances differ by more than
float64 rounding."""
import numpy as np
import pytest
import torch

from f2cgt_amd import capi

pytestmark = pytest.mark.gpu


def labels64(x, c, metric):
    x, c = x.astype(np.float64), c.astype(np.float64)
    with np.errstate(invalid="ignore"):
        if metric == "cosine":
            den = np.linalg.norm(x, axis=1)[:, None] * np.linalg.norm(c, axis=1)[None]
            d = 1.0 - (x @ c.T) / np.maximum(den, 1e-8)
        else:
            d = ((x[:, None] - c[None]) ** 2).sum(-1)
    d = np.where(np.isfinite(d), d, np.inf)
    two = np.partition(d, 1, axis=1)[:, :2] if c.shape[0] > 1 else np.stack([d[:, 0], d[:, 0] + 1], 1)
    two = np.minimum(two, np.finfo(np.float64).max)
    near = two[:, 1] - two[:, 0] <= 1e-12 * (1.0 + np.abs(two[:, 0]))        # float64 sums in another order
    return d.argmin(1), near


def check(x, c, metric):
    want, near = labels64(x, c, metric)
    got = capi.kmeans_predict(torch.from_numpy(x).cuda(), torch.from_numpy(c).cuda(), metric).cpu().numpy()
    assert np.array_equal(got[~near], want[~near])
    assert ((got >= 0) & (got < c.shape[0])).all()
    return near


# n: one tile, one centre, full and ragged last tiles, chunks of an odd number of tiles, several chunks;
# k: operand steps from 1 to 4 and both sides of each, rows that end in every mix of fours, twos and ones;
# m: a group of 32 rows, one less, one more, more groups than a workgroup has waves
@pytest.mark.parametrize("metric", ["cosine", "l2"])
@pytest.mark.parametrize("m,n,k", [
    (1, 1, 1), (31, 2, 3), (32, 31, 4), (33, 32, 7), (400, 33, 8), (500, 64, 9), (1000, 65, 15), (2000, 96, 16), (700, 97, 17),
    (300, 128, 22), (300, 129, 31), (3000, 160, 32), (500, 161, 33), (500, 256, 47), (500, 200, 48), (500, 65, 49), (500, 63, 61),
    (9000, 256, 64), (700, 1000, 16), (300, 1, 40), (600, 30, 5)])
def test_labels_are_the_first_minimum(metric, m, n, k):
    print("case assign", metric, m, n, k, flush=True)
    rng = np.random.default_rng(m * 7 + n * 3 + k)
    check(rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((n, k)).astype(np.float32), metric)


# rows and centres of very different lengths, down to where products vanish and up to where squares overflow, and data
# far from the origin: the scales of the pieces, the mean and the exact evaluation
@pytest.mark.parametrize("metric", ["cosine", "l2"])
@pytest.mark.parametrize("spread,centre_scale,shift", [(8, 1.0, 0.0), (0, 1e-12, 0.0), (0, 1e15, 0.0), (3, 1.0, 50.0), (18, 1e18, 0.0)])
@pytest.mark.parametrize("k", [16, 30])
def test_labels_over_scales(metric, spread, centre_scale, shift, k):
    print("case assign scales", metric, spread, centre_scale, shift, k, flush=True)
    rng = np.random.default_rng(k + spread)
    x = rng.standard_normal((600, k)) * 10.0 ** rng.uniform(-spread, spread, (600, 1)) + shift
    c = (rng.standard_normal((140, k)) + shift) * centre_scale
    x, c = x.astype(np.float32), c.astype(np.float32)
    if metric == "cosine":        # the clamp of |x||c| at 1e-8 makes float64 ties of its own
        x = x[np.linalg.norm(x.astype(np.float64), axis=1) * np.linalg.norm(c.astype(np.float64), axis=1).min() > 1e-7]
    if len(x):
        check(x, c, metric)


# a centre that is no number is never the nearest, wherever its tile and slot, and takes no other one of its class along
@pytest.mark.parametrize("metric", ["cosine", "l2"])
@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("n,bad", [(256, (0, 37, 255)), (40, (33,)), (20, (3,))])
def test_centres_that_are_no_numbers(metric, value, n, bad):
    print("case assign bad centres", metric, value, n, flush=True)
    rng = np.random.default_rng(n)
    x, c = rng.standard_normal((500, 16)).astype(np.float32), rng.standard_normal((n, 16)).astype(np.float32)
    for b in bad:
        c[b, b % 16] = value
    check(x, c, metric)


@pytest.mark.parametrize("metric", ["cosine", "l2"])
def test_rows_that_are_no_numbers(metric):
    rng = np.random.default_rng(3)
    x, c = rng.standard_normal((200, 24)).astype(np.float32), rng.standard_normal((100, 24)).astype(np.float32)
    x[5, 3], x[64, 0], x[199, 23] = np.nan, np.inf, -np.inf
    near = check(x, c, metric)
    assert near.sum() <= 3 + 1


# squares beyond the largest float, of some centres or of all, with rows beside the large centres and far from them: neither
# the scores nor the fp32 distances hold a number, and float64 on the original values decides
@pytest.mark.parametrize("metric", ["cosine", "l2"])
@pytest.mark.parametrize("scale", [1e20, 1.5e20, 1e21, 1e25, 1e30, 1e36])
@pytest.mark.parametrize("large", ["one", "half", "all"])
@pytest.mark.parametrize("k", [1, 16, 30, 64])
def test_values_whose_squares_overflow(metric, scale, large, k):
    print("case assign overflow", metric, scale, large, k, flush=True)
    rng = np.random.default_rng(k)
    n = 300 if k == 16 else 140
    c = rng.standard_normal((n, k))
    pick = {"one": [n - 3], "half": list(range(0, n, 2)), "all": list(range(n))}[large]
    c[pick] *= scale
    x = rng.standard_normal((500, k))
    x[::2] *= scale
    x[:n] = np.where(np.arange(n)[:, None] % 3 == 0, c * 1.0001, x[:n])
    check(x.astype(np.float32), c.astype(np.float32), metric)


# cosine: rows whose fp32 dot products overflow, in every order of signs
@pytest.mark.parametrize("size", [1e38, 3.3e38])
@pytest.mark.parametrize("k", [4, 16, 50])
def test_rows_whose_products_overflow(size, k):
    print("case assign overflow rows", size, k, flush=True)
    rng = np.random.default_rng(k)
    x = (np.sign(rng.standard_normal((300, k))) * size * rng.uniform(0.5, 1.0, (300, k))).astype(np.float32)
    check(x, rng.standard_normal((70, k)).astype(np.float32), "cosine")


# cosine: rows so short that their squares vanish in fp32, against centres so long that |x||c| stays above the clamp at 1e-8
@pytest.mark.parametrize("short", [18.5, 19.5, 21, 23, 26, 30, 36])
@pytest.mark.parametrize("k", [3, 16, 30, 64])
def test_rows_whose_squares_vanish(short, k):
    print("case assign short rows", short, k, flush=True)
    rng = np.random.default_rng(k)
    x = rng.standard_normal((600, k)) * 10.0 ** -short
    x[::50] = 0
    c = rng.standard_normal((140, k)) * 1e31
    near = check(x.astype(np.float32), c.astype(np.float32), "cosine")
    assert near.sum() < 40


# the same against centres of ordinary length, where the clamp makes the float64 distances equal: the label is that of the
# row's direction, which a power of two does not change
@pytest.mark.parametrize("power", [50, 62, 63, 64, 66, 80, 100, 110, 120, 130])
@pytest.mark.parametrize("k", [3, 16, 30, 64])
def test_rows_whose_squares_vanish_keep_their_direction(power, k):
    print("case assign short direction", power, k, flush=True)
    rng = np.random.default_rng(k)
    c = rng.standard_normal((140, k)).astype(np.float32)
    c[139], c[100], c[60] = c[7], 2 * c[20], c[61] * np.float32(1 + 1e-6)       # ties, decided in float64 among them alone
    to = rng.integers(0, 140, 700)
    x = (c[to] * rng.uniform(0.5, 2, (700, 1)) + 0.01 * rng.standard_normal((700, k))).astype(np.float32)
    want, _ = labels64(x, c, "cosine")
    d = 1 - (x / np.linalg.norm(x, axis=1)[:, None]).astype(np.float64) @ (c / np.linalg.norm(c, axis=1)[:, None]).astype(np.float64).T
    clear = np.partition(d, 1, axis=1)[:, :2] @ [-1, 1] > 1e-3
    zero = np.zeros(700, bool)
    zero[1::50] = True
    x[::3] *= np.float32(2.0 ** -(power - 20)) * np.float32(2.0 ** -20)         # beside rows of ordinary length
    x[zero] = 0
    got = capi.kmeans_predict(torch.from_numpy(x).cuda(), torch.from_numpy(c).cuda(), "cosine").cpu().numpy()
    assert np.array_equal(got[clear & ~zero], want[clear & ~zero]) and clear.sum() > 300
    # (3e-4: what rows of 2^-130 have left of their values, and products of theirs)
    assert (d[np.arange(700), got] - d.min(1))[~zero].max() < 3e-4
    assert (got[zero] == 0).all()                   # a row of zeros is as far from every centre


@pytest.mark.parametrize("metric", ["cosine", "l2"])
@pytest.mark.parametrize("m", [1, 31, 33, 70])
def test_rows_at_the_end_of_a_table_at_every_width(metric, m):
    """The last groups' rows, whose ends are read from inside the row: every length of the chunk of eight that a row ends in."""
    rng = np.random.default_rng(m)
    for k in range(1, 65):
        check(rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((70, k)).astype(np.float32), metric)
