"""1-bit log-domain rows with one codebook: items of eight columns, exchanged between the halves of a wave before they are
stored.  The same values in the same order as decoding the rows and aggregating them, so bit for bit the same."""
import pytest

torch = pytest.importorskip("torch")

if torch.cuda.is_available():
    from f2cgt_amd import capi, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim", [64, 66, 68, 70, 72, 130, 254, 602, 1030])
@pytest.mark.parametrize("rows,longest", [(1, 5), (7, 20), (9, 1), (300, 20), (2050, 6), (40, 900)])
@pytest.mark.parametrize("mode", ["stream", "cached"])
def test_equal_to_decode_and_aggregate(dim, rows, longest, mode):
    g = torch.Generator(device="cuda")
    g.manual_seed(dim * 1000 + rows)
    n = 501
    codes = torch.randint(-128, 128, (n, (dim + 7) // 8), generator=g, device="cuda", dtype=torch.int8)
    book = torch.tensor([[0.006, 2.8, -7.38, 1.485, 0.8123]], device="cuda")
    width = (dim + 7) // 8 * 8
    decoded = capi.sq_decompress(codes, book, 1, width, dim)
    deg = torch.randint(0, longest + 1, (rows,), generator=g, device="cuda")
    deg[0] = longest
    for dtype in (torch.int64, torch.int32):
        indptr = synth.csc_from_degrees(deg, dtype)
        indices = torch.randint(0, n, (int(indptr[-1]),), generator=g, device="cuda").to(dtype)
        want = capi.spmm_csr(decoded, indptr, indices)
        room = torch.full((rows + 8, dim), 5.0, device="cuda")      # four guard rows on either side
        was = capi.set_store_mode(capi.STORE_STREAM if mode == "stream" else capi.STORE_CACHED)
        try:
            capi.sq_decompress_spmm_csr(codes, book, indptr, indices, 1, width, dim, out=room[4:rows + 4])
        finally:
            capi.set_store_mode(was)
        assert torch.equal(room[4:rows + 4], want)
        assert bool((room[:4] == 5.0).all()) and bool((room[rows + 4:] == 5.0).all())
