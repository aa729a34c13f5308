"""Decode through a row list against fetch and decode, bit for bit: every id type, both widths of rows, remainders of the
row steps, ids outside the table, and the seed lookup with its errors."""
import pytest
import torch

import f2cgt_amd
from f2cgt_amd import pipeline

pytestmark = pytest.mark.gpu


def ids(n, rows, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    index = torch.randint(0, rows, (n,), generator=g)
    index[0], index[n // 2], index[-1] = rows + 5, -3, rows - 1       # held to the table like a fetch's
    return index.to(dtype).cuda()


# n: below the row list's kernel, its smallest, one step more or less, several steps per workgroup; dim: one tile and two,
# ragged, 4 k + 2 columns, odd (left to fetch and decode)
@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("n,dim,w,k", [
    (5, 128, 16, 256), (1023, 64, 8, 256), (1024, 64, 8, 256), (1025, 66, 4, 17), (1279, 128, 32, 256), (1281, 130, 16, 200),
    (70000, 100, 4, 256), (200000, 128, 16, 256), (5000, 256, 128, 9), (3000, 97, 8, 256), (2000, 100, 20, 256)])
def test_vq_rows(n, dim, w, k, dtype):
    print("case vq_rows", n, dim, w, k, dtype, flush=True)
    lib = f2cgt_amd.load()
    books = (dim + w - 1) // w
    g = torch.Generator(device="cuda").manual_seed(n)
    table = torch.randint(0, 256, (9001, books), generator=g, device="cuda", dtype=torch.uint8)
    cb = torch.randn((books, k, w), generator=g, device="cuda")
    index = ids(n, 9001, dtype, n)
    assert torch.equal(lib.vq_decompress_rows(table, index, cb, dim), lib.vq_decompress(lib.fetch_rows(table, index), cb, dim))


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("bits", [1, 2, 4, 8])
@pytest.mark.parametrize("n,dim,slice_", [(1, 8, 8), (7, 10, 16), (1025, 128, 128), (3, 602, 608), (4001, 100, 32), (900, 30, 8), (64, 7, 8),
                                          (2049, 8, 8), (3001, 10, 16), (5001, 154, 160),    # most rows to a workgroup; an odd count of them
                                          (501, 530, 10), (501, 540, 10), (501, 610, 10), (501, 620, 10)])   # 8 bits: both sides of the LDS budget
def test_sq_rows(n, dim, slice_, bits, dtype):
    print("case sq_rows", n, dim, slice_, bits, dtype, flush=True)
    lib = f2cgt_amd.load()
    g = torch.Generator(device="cuda").manual_seed(n)
    table = torch.randint(-128, 128, (5003, (dim * bits + 7) // 8), generator=g, device="cuda", dtype=torch.int8)
    n_cb = (dim + slice_ - 1) // slice_
    cb = torch.tensor([[0.01, 3.0, -6.6, 1.6 + 0.1 * i, 0.8] for i in range(n_cb)], device="cuda")
    index = ids(n, 5003, dtype, n) if n > 1 else torch.tensor([4999], dtype=dtype).cuda()
    want = lib.sq_decompress(lib.fetch_rows(table, index), cb, bits, slice_, dim)
    assert torch.equal(lib.sq_decompress_rows(table, index, cb, bits, slice_, dim), want)


@pytest.mark.parametrize("dim,bits", [(100, 4), (128, 8), (602, 4), (7, 4)])
@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
def test_seed_lookup(dim, bits, dtype):
    slice_ = (dim + 7) // 8 * 8
    g = torch.Generator(device="cuda").manual_seed(dim)
    seeds = torch.randperm(4000, generator=g, device="cuda")[:600]
    manager = pipeline.CompressionManager(
        {"methods": ["sq", "vq"], "feat_dim": dim, "configs": [(slice_, bits), (8, -1)],
         "codebooks": [torch.tensor([[0.01, 3.0, -6.6, 1.6, 0.8]], device="cuda"), torch.randn(((dim + 7) // 8, 16, 8), device="cuda")],
         "compression_data": torch.randint(0, 16, (4000, (dim + 7) // 8), device="cuda", dtype=torch.uint8),
         "seeds_compression_data": torch.randint(-128, 128, (600, (dim * bits + 7) // 8), generator=g, device="cuda", dtype=torch.int8),
         "seeds": seeds}, fusion=True)
    pick = torch.randint(0, 600, (333,), generator=g, device="cuda")
    want = manager._decompress(0, manager.seeds_data[pick])
    keys = seeds[pick].to(dtype)
    keys[7] -= 4000                                        # from the end, as an index is
    got = manager.get_seeds_data(keys)
    torch.cuda.current_stream().wait_event(manager.seeds_task_event)
    assert torch.equal(got, want)
    other = torch.ones(4000, dtype=torch.bool, device="cuda")
    other[seeds] = False
    keys[5] = torch.nonzero(other)[0, 0]
    with pytest.raises(KeyError):
        manager.get_seeds_data(keys)
    manager.check_seed_keys = False
    got = manager.get_seeds_data(keys)
    torch.cuda.synchronize()
    assert torch.equal(got[6:], want[6:]) and torch.equal(got[5], manager._decompress(0, manager.seeds_data[pick[:1] * 0])[0])


# 7 columns: looked up with torch, fetched and decoded
@pytest.mark.parametrize("dim", [8, 7])
def test_ids_outside_the_seed_map(dim):
    lib = f2cgt_amd.load()
    table = torch.arange(80, dtype=torch.int8, device="cuda").view(10, 8)[:, :dim].contiguous()
    slots = torch.arange(10, dtype=torch.int32, device="cuda")
    slots[3] = -1
    cb = torch.tensor([[0.01, 3.0, -6.6, 1.6, 0.8]], device="cuda")
    for bad in (10, -11, 2 ** 40):
        with pytest.raises(IndexError):
            lib.sq_decompress_rows(table, torch.tensor([1, bad, 2]).cuda(), cb, 8, 8, dim, slots, True)
        got = lib.sq_decompress_rows(table, torch.tensor([1, bad, -8]).cuda(), cb, 8, 8, dim, slots, False)
        assert torch.equal(got[::2], lib.sq_decompress(table[1:3], cb, 8, 8, dim)) and bool(torch.isfinite(got).all())
    with pytest.raises(KeyError):
        lib.sq_decompress_rows(table, torch.tensor([1, 3], dtype=torch.int32).cuda(), cb, 8, 8, dim, slots, True)
    empty = torch.empty((0,), dtype=torch.int64, device="cuda")
    assert lib.sq_decompress_rows(table, empty, cb, 8, 8, dim, slots, True).shape == (0, dim)
