"""Which calls take which kernels, where a rule on their sizes decides (no device needed)."""
import ctypes

import pytest

from naiwa_moe import _lib


@pytest.mark.parametrize("rows,H,E,tiles", [
    (65, 8192, 126, False), (128, 8192, 128, False), (250, 5120, 60, False),   # twice as slow in tiles
    (65, 7168, 256, False), (688, 2048, 64, False), (512, 5120, 60, False), (2048, 8192, 8, False), (65, 2048, 512, False),
    (4032, 4096, 8, True), (4096, 4096, 8, True), (1024, 5120, 60, True), (2048, 4096, 32, True),
    (1999, 2048, 128, True), (512, 2048, 128, True), (512, 65024, 128, True), (512, 65032, 128, False),
    (629, 3840, 60, True), (512, 4096, 64, True), (1024, 4096, 32, True), (2048, 4096, 16, True),   # and in wave-per-row blocks
    (512, 2048, 64, False), (750, 2048, 64, True), (4125, 8192, 8, True), (4095, 8192, 3, False),
])
def test_router_tiles_by_logits(rows, H, E, tiles):
    """64-row tiles by the number of logits, where both kernels were timed, not by the hidden size."""
    lib = ctypes.CDLL(_lib.LIB_PATH)
    assert bool(lib.naiwa_router_row_tiles(rows, H, E, 1)) == tiles


@pytest.mark.parametrize("rows,H,E,tiles", [
    (512, 4096, 64, False), (2048, 4096, 16, True), (750, 2048, 64, False), (782, 2048, 64, True),
    (629, 3840, 60, True), (65, 7168, 256, False), (2050, 8192, 8, True), (512, 65032, 128, False),
])
def test_router_tiles_by_logits_of_f32_rows(rows, H, E, tiles):
    """f32 rows cost the tiles more: another line."""
    lib = ctypes.CDLL(_lib.LIB_PATH)
    assert bool(lib.naiwa_router_row_tiles(rows, H, E, 0)) == tiles


@pytest.mark.parametrize("n,slots,I,wide", [
    (64 * 128, 128, 768, False), (64 * 128 + 1, 128, 768, True),   # pairs an expert
    (1312, 16, 1024, False), (1312, 16, 2048, True),               # 128 and 256 blocks
    (4096 * 2, 8, 14336, True), (512 * 8, 66, 1408, False),
])
def test_prefill_tiles_by_pairs_and_blocks(n, slots, I, wide):
    lib = ctypes.CDLL(_lib.LIB_PATH)
    assert bool(lib.naiwa_prefill_wide_tiles(ctypes.c_int64(n), slots, I)) == wide
