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


@pytest.mark.parametrize("rows,width,slots,H,kparts,exact_q4,strips", [
    (4, 2, 8, 4096, 1, True, 1), (64, 2, 8, 4096, 1, True, 1), (4, 4, 60, 3072, 1, True, 1),      # up to 1.4 blocks a CU
    (16, 4, 60, 3072, 1, True, 2), (64, 2, 8, 4096, 7, True, 2), (64, 2, 16, 4096, 1, True, 2),
    (4, 4, 60, 3072, 1, False, 1), (64, 4, 32, 2560, 1, False, 1), (32, 4, 60, 2048, 1, False, 1),  # 2.5 and 3.3
    (64, 2, 16, 4096, 1, False, 2), (64, 2, 8, 6144, 2, False, 2), (5, 8, 66, 2048, 1, False, 2),   # 2, 3 and under 2
    (64, 2, 8, 4096, 7, False, 2), (8, 1, 1, 512, 1, False, 1), (1, 16, 4, 512, 1, False, 1),
])
def test_down_strips_by_blocks_a_cu(rows, width, slots, H, kparts, exact_q4, strips):
    lib = ctypes.CDLL(_lib.LIB_PATH)
    assert lib.naiwa_decode_mfma_down_strips(rows, width, slots, H, kparts, exact_q4) == strips
