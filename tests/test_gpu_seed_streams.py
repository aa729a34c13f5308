"""Seed rows of a two-level manager: with the check of the ids (made on the current stream) and without it (on a stream of
their own), requested from any stream, by several threads, and used on another one."""
import threading

import pytest

torch = pytest.importorskip("torch")

if torch.cuda.is_available():
    import f2cgt_amd
    from f2cgt_amd import pipeline

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def manager():
    g = torch.Generator(device="cuda")
    g.manual_seed(0)
    n, d = 5000, 64
    seeds = torch.randperm(n, generator=g, device="cuda")[:2000]
    meta = {"methods": ["sq", "vq"], "feat_dim": d, "configs": [(d, 4), (16, -1)],
            "codebooks": [torch.tensor([[0.01, 3.0, -6.6, 1.6, 0.8]]), torch.randn((4, 256, 16))],
            "compression_data": torch.randint(0, 256, (n, 4), generator=g, device="cuda", dtype=torch.uint8),
            "seeds_compression_data": torch.randint(-128, 128, (2000, d // 2), generator=g, device="cuda", dtype=torch.int8),
            "seeds": seeds}
    sm = pipeline.CompressionManager(meta, fusion=True)
    sm.want = f2cgt_amd.load().sq_decompress(sm.seeds_data.data, sm.codebooks[0], 4, d, d)
    sm.keys = seeds
    return sm


@pytest.mark.parametrize("check", [True, False])
@pytest.mark.parametrize("own_stream", [True, False])
def test_rows_from_any_stream(manager, check, own_stream):
    manager.check_seed_keys = check
    try:
        stream = torch.cuda.Stream() if own_stream else torch.cuda.current_stream()
        for i in range(5):
            pick = torch.randint(0, 2000, (700,), device="cuda")
            stream.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(stream):
                keys = manager.keys[pick] + 0                # still in the making when it is handed over
                rows = manager.get_seeds_data(keys)
                del keys
            other = torch.cuda.Stream()
            with torch.cuda.stream(other):
                got = manager.reorganize_seeds_data(rows, manager.get_all_data(manager.keys[:700]), 700)
            torch.cuda.synchronize()
            assert torch.equal(got, manager.want[pick])
            if check:
                free = torch.ones(5000, dtype=torch.bool, device="cuda")
                free[manager.keys] = False
                with pytest.raises(KeyError):
                    manager.get_seeds_data(torch.nonzero(free)[:3, 0])
    finally:
        manager.check_seed_keys = True


def test_rows_for_several_threads(manager):
    wrong = []

    def ask(seed):
        g = torch.Generator(device="cuda")
        g.manual_seed(seed)
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(20):
                pick = torch.randint(0, 2000, (300,), generator=g, device="cuda")
                rows = manager.get_seeds_data(manager.keys[pick])
                if not torch.equal(rows, manager.want[pick]):
                    wrong.append(seed)

    threads = [threading.Thread(target=ask, args=(s,)) for s in range(4)]
    torch.cuda.synchronize()
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


@pytest.mark.parametrize("check", [True, False])
def test_keys_on_the_host_are_refused(manager, check):
    manager.check_seed_keys = check
    try:
        with pytest.raises(RuntimeError):
            manager.get_seeds_data(manager.keys[:10].cpu())
    finally:
        manager.check_seed_keys = True
