"""The gather by one block an expert id: bit-exact at the edges of its register sizes, ids
outside the range counted and left out."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,E", [(257, 3), (4096, 64), (4097, 64), (8193, 128), (16385, 60), (40000, 8),
                                 (65536, 128)])
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
