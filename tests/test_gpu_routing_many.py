"""Router logits of many rows in 64-row tiles: bit-exact against the oracle at the edges of the
tiles."""
import numpy as np
import pytest

import oracle as O
import synthetic as S
from test_gpu_routing import gpu_router

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,H,E,x_f32", [
    (512, 2048, 128, False),   # whole tiles
    (450, 512, 129, False),    # a ragged row tile and expert group
    (1090, 520, 61, False),    # a part of a unit at the end of K
    (8200, 64, 8, False),      # one unit: seven of the eight waves have none
    (1000, 1032, 66, True),    # f32 rows, a part of a unit
    (65, 8192, 126, False),    # few logits at a large H: not in tiles
])
def test_many_row_logits_bit_exact(gpu, rows, H, E, x_f32):
    x = S.activations_bf16(4200 + rows, rows, H)
    W = O.normal(4201 + E, E * H, 0.0, 0.02).reshape(E, H)
    print(f"[router rows={rows} H={H} E={E} f32={x_f32}]", flush=True)
    ids, _, logits = gpu_router(gpu, x, W, 4, O.ROUTE_TOPK_SOFTMAX, x_f32=x_f32)
    want = O.router_logits(O.from_bf16(x), W)
    assert np.array_equal(logits.view(np.uint32), want.view(np.uint32))
    assert np.array_equal(ids, O.topk(want, 4, O.ROUTE_TOPK_SOFTMAX)[0])


def test_many_row_logits_of_large_chunks(gpu):
    """Chunks past the fast rounding's range of 2^12 (and sums past it), beside ordinary rows."""
    rows, H, E = 1024, 512, 64
    xs = O.from_bf16(S.activations_bf16(4300, rows, H)).copy()
    xs[::3] *= np.float32(2.0 ** 17)
    xs[1::3] *= np.float32(2.0 ** 11)
    x = O.to_bf16(xs)
    W = O.normal(4301, E * H, 0.0, 0.02).reshape(E, H)
    _, _, logits = gpu_router(gpu, x, W, 4, O.ROUTE_TOPK_SOFTMAX)
    want = O.router_logits(O.from_bf16(x), W)
    assert np.abs(want[::3]).max() > 2.0 ** 12
    assert np.array_equal(logits.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("H", [65024, 65088, 65472])   # the largest in 64-row tiles, and past it
@pytest.mark.parametrize("x_f32", [False, True])
def test_many_row_logits_of_half_way_chunks(gpu, H, x_f32):
    """Every chunk is 2^-11, where the low part of the split rounding is largest: the low sums of
    a wave's chunks still fit 32 bits at the longest rows the tiles take."""
    rows, E = 512, 128
    x = np.full((rows, H), 0x3F80, np.uint16)                       # 1.0
    W = np.full((E, H), np.float32(2.0 ** -14), np.float32)
    _, _, logits = gpu_router(gpu, x, W, 4, O.ROUTE_TOPK_SOFTMAX, x_f32=x_f32)
    assert np.all(logits == np.float32(H * 2.0 ** -14))
