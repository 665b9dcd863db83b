"""Prefill's 128-pair tiles (calls that average more than 64 pairs an expert and give every CU a
block): segments at every edge of the 32-row subtiles, in all four format pairs, bit for bit
against the same rows in calls of few pairs an expert (64-pair tiles): an output row depends on
its own token alone, and both kernels round the same values.  Some rows of every expert are
also held against the oracle."""
import ctypes

import numpy as np
import pytest

import oracle as O
import synthetic as S
from naiwa_moe import _lib

pytestmark = pytest.mark.gpu

# pairs of each expert: one, around each subtile, whole tiles, splits of 2 and 3 tiles, none
COUNTS = [1, 31, 32, 33, 64, 65, 97, 128, 129, 160, 193, 257, 300, 0, 96, 2]


def takes_wide_tiles(n, slots, I):
    return bool(ctypes.CDLL(_lib.LIB_PATH).naiwa_prefill_wide_tiles(ctypes.c_int64(n), slots, I))


@pytest.mark.parametrize("H,I,dt", [
    (256, 2048, (O.Q4_K, O.Q4_K, O.Q4_K)),    # one K-block of gate/up
    (768, 2176, (O.Q4_K, O.Q4_K, O.Q8_0)),    # an odd number of K-blocks each way
    (256, 2304, (O.Q8_0, O.Q8_0, O.Q4_K)),
    (512, 2176, (O.Q8_0, O.Q8_0, O.Q8_0)),
])
def test_wide_tiles(gpu, H, I, dt):
    nm = gpu
    E, T = len(COUNTS), sum(COUNTS)
    assert takes_wide_tiles(T, E, I) and not takes_wide_tiles(64 * E, E, I)
    g, u, d, _ = S.layer(4100 + H, E, H, I, dt)
    banks = nm.LayerBanks(E, H, I, dt)
    for e in range(E):
        banks.load(e, g[e], u[e], d[e])
    rng = np.random.default_rng(H + I)
    ids = rng.permutation(np.repeat(np.arange(E), COUNTS)).astype(np.uint32).reshape(T, 1)
    w = rng.uniform(0.1, 1.0, (T, 1)).astype(np.float32)
    x = S.activations_bf16(4101 + I, T, H)

    def call(rows):
        out = nm.DeviceBuffer(len(x[rows]) * H * 4)
        xd, idd, wd = (nm.DeviceBuffer.from_array(np.ascontiguousarray(a[rows])) for a in (x, ids, w))
        nm.moe_prefill(banks, xd, idd, wd, len(x[rows]), 1, out)
        nm.synchronize()
        return out.download(np.float32).reshape(-1, H)

    print(f"[prefill wide H={H} I={I} dt={dt}]", flush=True)
    got = call(slice(0, T))
    few = np.concatenate([call(slice(t, min(T, t + 64 * E))) for t in range(0, T, 64 * E)])
    assert np.array_equal(got.view(np.uint32), few.view(np.uint32))
    some = np.concatenate([np.nonzero(ids[:, 0] == e)[0][[0, -1]] for e in range(E) if COUNTS[e]])
    want = O.fused_moe_decode(O.stack(g, dt[0], I, H), O.stack(u, dt[1], I, H), O.stack(d, dt[2], H, I),
                              O.from_bf16(x[some]), ids[some], w[some])
    assert S.max_rel_err(got[some], want) < 1e-2   # bf16 weights and h, as for the 64-pair tiles

