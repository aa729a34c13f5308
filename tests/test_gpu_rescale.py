"""Centres rescaled to their slice's mean length in one launch, against float64; its flags; and what vq_metadata raises."""
import pytest

torch = pytest.importorskip("torch")

if torch.cuda.is_available():
    import f2cgt_amd
    from f2cgt_amd import pipeline

pytestmark = pytest.mark.gpu


def _codebooks(centers, bad=None):
    """The loop with no step to make, so that the centres are the ones given."""
    x = torch.randn((centers.shape[0], 64, centers.shape[2]), device="cuda")
    return f2cgt_amd.load().kmeans_slices_fit(x, None, centers, "cosine", 2, 5e-2, 1.2, 0, 8, bad, True)


@pytest.mark.parametrize("slices,n,k", [(1, 1, 1), (3, 16, 8), (6, 256, 16), (2, 257, 33), (1, 512, 64)])
def test_lengths_and_directions(slices, n, k):
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    c = torch.randn((slices, n, k), generator=g, device="cuda") * torch.rand((slices, n, 1), generator=g, device="cuda") * 10
    flags, books = _codebooks(c.clone(), torch.ones((1,), dtype=torch.int32, device="cuda"))
    C = c.double()
    norms = C.norm(dim=2, keepdim=True)
    want = C / norms * norms.mean(dim=1, keepdim=True)
    # a length, its mean, a quotient and a product, each rounded once
    assert bool(((books.double() - want).abs() <= 5 * 2.0 ** -24 * want.abs()).all())
    assert flags.tolist() == [0] * slices + [1, 0]


def test_flags_and_errors():
    c = torch.ones((2, 4, 8), device="cuda")
    c[1, 2] = 0                                   # a centre without a length
    assert _codebooks(c)[0].tolist() == [0, 0, 0, 1]
    x = torch.randn((2000, 20), device="cuda")
    torch.manual_seed(0)
    books = pipeline.vq_metadata(x, 16, 8, sample_index=torch.arange(2000), max_iter=4)
    assert books.shape == (3, 16, 8) and bool((books[2, :, 4:] == 0).all())
    with pytest.raises(IndexError):
        pipeline.vq_metadata(x, 16, 8, sample_index=torch.tensor([0, 5, 2000] * 100), max_iter=4)
    x[3, 1] = float("nan")
    with pytest.raises(RuntimeError, match="no rows"):
        pipeline.vq_metadata(x, 16, 8, sample_index=torch.arange(2000), max_iter=4)
