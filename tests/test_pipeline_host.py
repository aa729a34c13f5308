"""Host-side pieces of f2cgt_amd/pipeline.py that need no GPU."""
import types

import numpy as np
import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

import f2cgt_oracle as oc
from f2cgt_amd import pipeline


def test_sq_metadata_is_the_reference_codebook_statement():
    rng = np.random.default_rng(0)
    for scale, shift in ((1.0, 0.0), (1e-4, 0.0), (3.0, 10.0)):
        x = (rng.standard_normal((5000, 7)) * scale + shift).astype(np.float32)
        got = np.array([float(v) for v in pipeline.sq_metadata(torch.from_numpy(x))], dtype=np.float32)
        want = oc.sq_codebook(x)
        assert np.array_equal(got[:4], want[:4])
        assert np.isclose(got[4], want[4], rtol=1e-6)


def test_log2_of_a_codebook_is_correctly_rounded():
    """As the device makes it, so that sq_metadata and sq_compress agree on the same sample."""
    values = np.exp(np.random.default_rng(1).uniform(np.log(1e-5), np.log(1e3), 20000)).astype(np.float32)
    want = np.log2(values.astype(np.float64)).astype(np.float32)
    got = [pipeline._sq_codebook(v, v, torch.tensor(1.0)) for v in values]
    assert np.array_equal([np.float32(b[2]) for b in got], want)
    top = np.log2(np.maximum(values, np.float32(2e-5)).astype(np.float64)).astype(np.float32) + np.float32(1e-5)
    assert np.array_equal([np.float32(b[3]) for b in got], top)


def test_normalize_rescales_rows_to_the_mean_norm():
    x = torch.tensor([[3.0, 4.0], [0.0, 1.0], [6.0, 8.0]])
    y = pipeline.normalize(x)
    mean_norm = (5.0 + 1.0 + 10.0) / 3.0
    assert torch.allclose(y.norm(dim=1), torch.full((3,), mean_norm))
    assert torch.allclose(y[0] / y[0].norm(), x[0] / x[0].norm())


def test_sampling_is_a_permutation_prefix_or_follows_hotness():
    g = torch.Generator().manual_seed(3)
    s = pipeline.sampling(10, 100, generator=g)
    assert s.numel() == 10 and s.unique().numel() == 10 and int(s.max()) < 100
    np.random.seed(0)
    hot = torch.zeros(50)
    hot[:5] = 1.0
    s = pipeline.sampling(5, 50, hotness=hot)
    assert sorted(s.tolist()) == [0, 1, 2, 3, 4]


def test_layer_rejects_other_aggregators():
    import pytest
    with pytest.raises(ValueError):
        pipeline.MySAGEConv(8, 4, "pool", None)


def test_what_the_device_statistics_take():
    """The sizes that sq_compress keeps from the device statistics are those that the library refuses (its checks come
    before anything is read: the buffers are stand-ins)."""
    import ctypes
    from f2cgt_amd import capi
    a, ranks = ctypes.c_void_p(1 << 20), (ctypes.c_int64 * 8)()
    assert pipeline._device_takes(1, 1, 1) and pipeline._device_takes(2 ** 32 - 1, 1, 1)
    assert pipeline._device_takes(5, 2 ** 24 - 1, 300) and pipeline._device_takes(3, 65535, 1)
    for m, cols, width in ((2 ** 32, 1, 1), (2 ** 25, 500, 128), (3, 2 ** 24, 2 ** 24), (3, 65536, 1), (0, 8, 8), (8, 0, 8)):
        assert not pipeline._device_takes(m, cols, width)
        assert capi.lib().f2cgt_abs_order_stats(a, max(cols, 1), a, m, max(m, 1), cols, width, ranks, a, 1 << 62, a, None)


class _Devices:
    """Stands for the operator library: checks that the tensors of a call lie on one device, computes nothing."""

    def __init__(self):
        self.calls = []

    def sq_codebooks(self, x, rows, column_slice, ranks, weights):
        self.calls.append("sq_codebooks")
        assert rows.device == x.device
        slices = -(-x.shape[1] // column_slice)
        stats = types.SimpleNamespace(cpu=lambda: types.SimpleNamespace(numpy=lambda: np.zeros((slices, 6))))
        return torch.empty((slices, 5), device=x.device), stats

    def sq_encode(self, data, codebooks, bits, column_slice, out):
        self.calls.append("sq_encode")
        assert data.device == codebooks.device == out.device

    def kmeans_slices_covers(self, slices, n, k):
        return True

    def slice_rows(self, x, rows, column_slice):
        assert rows is None or rows.device == x.device
        m, slices = (x.shape[0] if rows is None else rows.numel()), -(-x.shape[1] // column_slice)
        return (torch.empty((slices, m, column_slice), device=x.device), torch.empty((m, slices), device=x.device),
                torch.empty((1,), device=x.device, dtype=torch.int32))

    def abs_order_stats(self, x, rows, column_slice, ranks):
        return torch.empty((x.shape[1], 6), device=x.device, dtype=torch.float64)

    def keep_rows(self, norms, stats, weight, weight_last):
        return torch.empty((norms.shape[1], -(-norms.shape[0] // 32)), device=norms.device, dtype=torch.int32)

    def kmeans_slices_fit(self, data, keep, centers, *rest):
        self.calls.append("kmeans_slices_fit")
        assert data.device == keep.device == centers.device
        raise StopIteration


@pytest.mark.parametrize("table", ["cuda:0", "cuda:1"])
def test_sq_codes_of_a_table_on_a_device_that_is_not_the_current_one(table, monkeypatch):
    """Codes and codebooks are made on the current device, wherever the table lies."""
    lib = _Devices()
    monkeypatch.setattr(pipeline, "_capi", lambda: lib)
    with FakeTensorMode():
        x = torch.empty((1000, 40), device=table)
        codes, books = pipeline.sq_compress(x, 4, 16, sample_index=torch.arange(500))
        assert str(codes.device) == str(books.device) == "cuda:0"
    assert lib.calls == ["sq_codebooks", "sq_encode"]


@pytest.mark.parametrize("table", ["cuda:0", "cuda:1"])
def test_codebooks_of_a_table_on_a_device_that_is_not_the_current_one(table, monkeypatch):
    lib = _Devices()
    monkeypatch.setattr(pipeline, "_capi", lambda: lib)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    with FakeTensorMode():
        x = torch.empty((1000, 40), device=table)
        with pytest.raises(StopIteration):
            pipeline._train_all_slices(x, 16, 8, torch.arange(500), 4)
    assert lib.calls == ["kmeans_slices_fit"]
