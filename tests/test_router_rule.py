"""Which router calls take 64-row tiles (no device needed): by their number of logits, where
both kernels were measured, and not by the hidden size."""
import ctypes

import pytest

from naiwa_moe import _lib


@pytest.mark.parametrize("rows,H,E,tiles", [
    (65, 8192, 126, False), (128, 8192, 128, False), (250, 5120, 60, False),   # twice as slow in tiles
    (65, 7168, 256, False), (512, 5120, 60, False), (2048, 8192, 8, False), (65, 2048, 512, False),
    (4032, 4096, 8, True), (4096, 4096, 8, True), (1024, 5120, 60, True), (2048, 4096, 32, True),
    (1999, 2048, 128, True), (512, 2048, 128, True), (512, 65024, 128, True), (512, 65032, 128, False),
])
def test_router_tiles_by_logits(rows, H, E, tiles):
    lib = ctypes.CDLL(_lib.LIB_PATH)
    assert bool(lib.naiwa_router_row_tiles(rows, H, E)) == tiles
