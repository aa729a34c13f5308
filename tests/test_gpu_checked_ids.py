"""sq_compress reads its sample's ids once, on the device, and waits for their check alone: what it raises and returns."""
import pytest

torch = pytest.importorskip("torch")

if torch.cuda.is_available():
    import f2cgt_amd
    from f2cgt_amd import pipeline

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,dim,slice_", [(300, 8, 8), (40000, 100, 104), (5000, 30, 8), (2000, 33, 33)])
def test_codebooks_and_flag(rows, dim, slice_):
    lib = f2cgt_amd.load()
    g = torch.Generator(device="cuda")
    g.manual_seed(rows)
    x = torch.randn((rows, dim), generator=g, device="cuda")
    for m in (1, 50, rows):
        ids = torch.randint(-rows, rows, (m,), generator=g, device="cuda")
        places = pipeline._percentile_places(m, dim, slice_)[1]
        ranks = [r for per_size in places for place in per_size for r in place[:2]]
        weights = [place[2] for per_size in places for place in per_size]
        want, stats = lib.sq_codebooks(x[ids], None, slice_, ranks, weights)
        assert not hasattr(stats, "bad_rows")
        for _ in range(3):                        # the workgroup that finishes last differs from run to run
            books, stats = lib.sq_codebooks(x, ids, slice_, ranks, weights)
            assert not stats.bad_rows.wait() and torch.equal(books, want) and not stats.bad_rows.wait()
        assert int(stats[:, 5].max()) == 0
        ids[m // 2] = rows
        assert lib.sq_codebooks(x, ids, slice_, ranks, weights)[1].bad_rows.wait()


def test_errors_and_calls_one_after_the_other():
    x = torch.randn((50000, 64), device="cuda")
    good = torch.randperm(50000, device="cuda")[:30000]
    bad = good.clone()
    bad[-1] = 50000
    want = pipeline.sq_compress(x, 4, 64, sample_index=good)
    torch.cuda.synchronize()
    for i in range(12):
        if i % 3 == 1:
            with pytest.raises(IndexError):
                pipeline.sq_compress(x, 4, 64, sample_index=bad)
        else:
            codes, books = pipeline.sq_compress(x, 4, 64, sample_index=good)
            assert torch.equal(books, want[1]) and torch.equal(codes, want[0])
    with pytest.raises(NotImplementedError):
        pipeline.sq_compress(x, 17, 64, sample_index=good)      # raised with the statistics still on their way


def test_codebooks_in_a_captured_graph():
    lib = f2cgt_amd.load()
    x = torch.randn((20000, 32), device="cuda")
    ids = torch.randint(0, 20000, (9000,), device="cuda")
    places = pipeline._percentile_places(9000, 32, 32)[1]
    ranks = [r for per_size in places for place in per_size for r in place[:2]]
    weights = [place[2] for per_size in places for place in per_size]
    make = lambda: lib.sq_codebooks(x, ids, 32, ranks, weights)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        make()[1].bad_rows.wait()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        books, stats = make()
    assert not hasattr(stats, "bad_rows")             # nothing waits during a capture
    for _ in range(4):
        x.normal_()
        ids.copy_(torch.randint(0, 20000, (9000,), device="cuda"))
        torch.cuda.synchronize()
        graph.replay()
        got = books.clone()
        assert torch.equal(got, make()[0])
