"""The gather by one block an expert id: bit-exact at the edges of its register sizes, ids
outside the range counted and left out."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,E", [(257, 3), (4096, 64), (4097, 64), (8193, 128), (16385, 60), (40000, 8),
                                 (65536, 128), (257, 4096), (1024, 4096), (1025, 2048), (2048, 300), (2049, 2048),
                                 (8192, 2048), (8193, 1000), (16384, 1024), (32768, 66), (32769, 500)])
def test_gather_by_id_bit_exact(gpu, n, E):
    nm = gpu
    rng = np.random.default_rng(n + E)
    ids = rng.integers(0, E, size=n).astype(np.uint32)
    ids[rng.integers(0, n, size=5)] = E + 7          # outside: counted, not placed
    nbad = int((ids >= E).sum())
    idsd, perm, off = nm.DeviceBuffer.from_array(ids), nm.DeviceBuffer(n * 4), nm.DeviceBuffer((E + 1) * 4)
    bad = nm.DeviceBuffer(4)
    nm.moe_gather(idsd, n, E, perm, off, bad)
    nm.synchronize()
    order = np.argsort(ids, kind="stable")[:n - nbad].astype(np.uint32)
    assert np.array_equal(perm.download(np.uint32, n - nbad), order)
    counts = np.bincount(ids[ids < E], minlength=E)
    assert np.array_equal(off.download(np.uint32), np.concatenate([[0], np.cumsum(counts)]).astype(np.uint32))
    assert bad.download(np.int32)[0] == nbad


def test_gather_of_few_entries_does_not_wait_for_idle_waves(gpu):
    """One block per id: with many ids and few entries, blocks of more waves than hold entries
    queue behind each other (three times the time of few ids' call, instead of about the same)."""
    nm = gpu
    n, times = 300, {}
    for E in (256, 4096):
        rng = np.random.default_rng(E)
        idsd = nm.DeviceBuffer.from_array(rng.integers(0, E, size=n).astype(np.uint32))
        perm, off = nm.DeviceBuffer(n * 4), nm.DeviceBuffer((E + 1) * 4)
        best = float("inf")
        for _ in range(8):
            start, stop = nm.Event(timing=True), nm.Event(timing=True)
            start.record(0)
            for _ in range(100):
                nm.moe_gather(idsd, n, E, perm, off)
            stop.record(0)
            nm.synchronize()
            best = min(best, start.elapsed_ms(stop))
        times[E] = best
    assert times[4096] < 2 * times[256]
