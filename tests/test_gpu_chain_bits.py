"""A layered step routes on its own rounded activations, so a change of a layer's rounding
flips an expert near the cut of a top-k somewhere: the bits of its matrix-core layers (4 rows
or more, at most 512 pairs) are pinned, as CRCs of the outputs that the first matrix-core
decode gave for the same seeded inputs."""
import zlib

import numpy as np
import pytest

import oracle as O
import synthetic as S

pytestmark = pytest.mark.gpu
Q4, Q8 = O.Q4_K, O.Q8_0


def step_crc(nm, dt, H, I, E, k, rows):
    """CRCs of y (f32) and of x + y (bf16) of a one-layer layered step."""
    g, u, d, r = S.layer(9100 + rows, E, H, I, dt)
    banks = nm.LayerBanks(E, H, I, dt)
    for e in range(E):
        banks.load(e, g[e], u[e], d[e])
    rd = nm.DeviceBuffer.from_array(r)
    desc = (nm._lib.Layer * 1)(nm.layer_desc(rd, banks))
    xd = nm.DeviceBuffer.from_array(S.activations_bf16(9101 + rows, rows, H))
    y = nm.DeviceBuffer(rows * H * 4)
    print(f"[chain bits {dt} H={H} I={I} E={E} k={k} rows={rows}]", flush=True)
    nm.stack_decode(desc, xd, rows, H, E, k, mode=O.ROUTE_SOFTMAX_TOPK_RENORM, fused=False, y_out=y)
    nm.synchronize()
    return zlib.crc32(y.download(np.uint32).tobytes()), zlib.crc32(xd.download(np.uint16).tobytes())


CASES = [
    ((Q4, Q4, Q4), 512, 512, 16, 4, 4),
    ((Q4, Q4, Q4), 512, 2304, 4, 2, 33),    # two K parts; chunks of 32 rows and past them
    ((Q4, Q4, Q8), 512, 384, 16, 4, 5),
    ((Q8, Q8, Q4), 384, 512, 16, 4, 17),
    ((Q8, Q8, Q8), 384, 128, 8, 4, 64),
    ((Q8, Q8, Q8), 512, 2176, 4, 2, 128),   # the last K part 128
    ((Q8, Q8, Q8), 1024, 640, 8, 8, 9),
    ((Q4, Q4, Q4), 2048, 256, 64, 8, 8),    # two strips of down rows a block
    ((Q4, Q4, Q8), 4096, 128, 32, 4, 11),   # one
    ((Q8, Q8, Q8), 2048, 128, 64, 8, 64),
    ((Q4, Q4, Q8), 4096, 128, 32, 4, 40),   # and in 16-row tiles
]
CRCS = [
    (0xD82292C2, 0x40582F51),
    (0x83FC265D, 0x3A45211C),
    (0xF62C3CA1, 0xAD18FD04),
    (0xED6EFDEA, 0x3D22C2A3),
    (0x1B1B5870, 0x5C0EC3A5),
    (0x6CF94595, 0x905DD976),
    (0x7D1449DF, 0xE654BB32),
    (0xC0AEE869, 0xC469268E),
    (0xA416CE1D, 0xC3613152),
    (0x31548153, 0x41809160),
    (0x4F544149, 0xFB8383EA),
]


@pytest.mark.parametrize("case,crc", list(zip(CASES, CRCS)))
def test_chain_bits(gpu, case, crc):
    assert step_crc(gpu, *case) == crc


@pytest.mark.parametrize("dt,E,k,rows", [
    ((Q4, Q4, Q4), 16, 4, 3),      # the GEMV kernels
    ((Q4, Q4, Q4), 16, 8, 65),     # 520 pairs: exact operands on both sides
    ((Q8, Q8, Q8), 16, 8, 70),
])
def test_layered_step_is_the_chain_of_the_public_calls(gpu, dt, E, k, rows):
    """Outside the rounded range a layered step gives the bits of naiwa_router_topk,
    naiwa_moe_decode and x = bf16(x + y)."""
    nm = gpu
    H, I = 256, 256
    layers = []
    for l in range(2):
        g, u, d, r = S.layer(9200 + l, E, H, I, dt)
        banks, rd = nm.LayerBanks(E, H, I, dt), nm.DeviceBuffer.from_array(r)
        for e in range(E):
            banks.load(e, g[e], u[e], d[e])
        layers.append((banks, rd))
    x = S.activations_bf16(9202, rows, H)
    xd = nm.DeviceBuffer.from_array(x)
    nm.stack_decode([nm.layer_desc(rd, b) for b, rd in layers], xd, rows, H, E, k,
                    mode=O.ROUTE_SOFTMAX_TOPK_RENORM, fused=False)
    ids, w, y = nm.DeviceBuffer(rows * k * 4), nm.DeviceBuffer(rows * k * 4), nm.DeviceBuffer(rows * H * 4)
    for banks, rd in layers:
        hd = nm.DeviceBuffer.from_array(x)
        nm.router_topk(hd, nm.BF16, rd, rows, H, E, k, ids, w, mode=O.ROUTE_SOFTMAX_TOPK_RENORM)
        nm.indexed_moe_fused_decode(banks, hd, nm.BF16, ids, w, rows, k, y)
        x = O.to_bf16(O.from_bf16(x) + y.download(np.float32).reshape(rows, H))
    assert np.array_equal(xd.download(np.uint16).reshape(rows, H), x)
