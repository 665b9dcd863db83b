"""The matrix-core decode (calls of 4 rows or more) against the oracle at the edges of its
tiles: 8-, 16- and 32-row activation tiles and chunks past them, one and two weight strips,
short last K parts, more than 512 pairs, rows of very different magnitudes, and the
no-alloc entry point's passes over the rows."""
import ctypes as C

import numpy as np
import pytest

import oracle as O
import synthetic as S

pytestmark = pytest.mark.gpu
Q4, Q8 = O.Q4_K, O.Q8_0
# Weights enter as exact integers with f32 scales, a bf16 x is kept exactly, h is rounded once to
# f16 (relative 2^-11 a value): a row's error stays below 2^-11 sum |h w| w_j, within 1e-3 of the
# largest output (f32 x is rounded to f16 as well: the same bound again).
TOL = 1e-3


def _layer(nm, seed, E, H, I, dt):
    g, u, d, r = S.layer(seed, E, H, I, dt)
    banks = nm.LayerBanks(E, H, I, dt)
    for e in range(E):
        banks.load(e, g[e], u[e], d[e])
    # the stacks point into the arrays: the caller keeps those
    return banks, (O.stack(g, dt[0], I, H), O.stack(u, dt[1], I, H), O.stack(d, dt[2], H, I)), (g, u, d)


@pytest.mark.parametrize("dt,H,I,E,k,rows,x_f32", [
    ((Q4, Q4, Q4), 256, 256, 4, 2, 4, False),       # one K-block each way
    ((Q4, Q4, Q8), 512, 384, 5, 3, 7, True),        # 8-row tile, odd rows, f32 x
    ((Q8, Q8, Q8), 384, 128, 3, 2, 9, False),       # 16-row tile
    ((Q8, Q8, Q4), 128, 512, 16, 2, 17, False),
    ((Q4, Q4, Q4), 256, 2304, 4, 2, 33, False),     # two K parts, the last 256; chunks of 32
    ((Q4, Q4, Q8), 256, 2176, 2, 1, 65, True),      # the last K part 128; segments past 32 rows
    ((Q4, Q4, Q4), 512, 256, 16, 8, 150, False),    # 1,200 pairs
    ((Q8, Q8, Q8), 256, 256, 8, 16, 40, False),     # 640 pairs, the widest row of pairs
    # one weight stage (more than a gate/up block a CU) in the 8- and 16-row tiles
    ((Q8, Q8, Q8), 256, 1152, 16, 2, 8, False),
    ((Q8, Q8, Q8), 384, 1152, 16, 2, 16, True),
    # several blocks along a segment: chunks past a block's first, blocks without one
    ((Q4, Q4, Q4), 256, 256, 2, 1, 50, False),      # 25 tokens a segment
    ((Q8, Q8, Q8), 256, 2304, 3, 2, 200, True),     # five blocks, two K parts
    ((Q4, Q4, Q8), 512, 128, 1, 1, 1000, False),    # 32 chunks
    # two strips of down rows a block (1,024 blocks of them), in each tile height
    ((Q4, Q4, Q4), 2048, 256, 64, 8, 8, False),
    ((Q4, Q4, Q8), 4096, 128, 32, 3, 11, False),
    ((Q4, Q4, Q4), 2048, 256, 64, 8, 70, False),
    ((Q8, Q8, Q8), 2048, 128, 64, 8, 70, True),
])
def test_exact_weights_at_tile_edges(gpu, dt, H, I, E, k, rows, x_f32):
    nm = gpu
    banks, stacks, keep = _layer(nm, 8100 + rows, E, H, I, dt)
    x = S.activations_bf16(8200 + rows, rows, H)
    xf = O.from_bf16(x)
    rng = np.random.default_rng(rows)
    ids = rng.integers(0, E, (rows, k)).astype(np.uint32)   # repeated slots among them
    w = rng.random((rows, k)).astype(np.float32)
    w[0, -1] = 0.0                                          # a padded pair
    if x_f32:
        xf = (xf * 1.0001).astype(np.float32)
    xd = nm.DeviceBuffer.from_array(xf if x_f32 else x)
    ids_d, w_d = nm.DeviceBuffer.from_array(ids), nm.DeviceBuffer.from_array(w)
    out = nm.DeviceBuffer(rows * H * 4)
    print(f"[mfma decode {dt} H={H} I={I} E={E} k={k} rows={rows}]", flush=True)
    nm.indexed_moe_fused_decode(banks, xd, nm.F32 if x_f32 else nm.BF16, ids_d, w_d, rows, k, out)
    got = out.download(np.float32).reshape(rows, H)
    err = S.max_rel_err(got, O.fused_moe_decode(*stacks, xf, ids, w))
    print(f"  max_rel_err={err:.3e}", flush=True)
    assert err < TOL


def test_rows_of_any_magnitude(gpu):
    nm = gpu
    E, H, I, k = 4, 256, 256, 2
    scales = np.array([0.0, 1e-12, 1e-3, 1.0, 1e6, 1e14], np.float32)
    banks, stacks, keep = _layer(nm, 8300, E, H, I, (Q4, Q4, Q4))
    x = O.to_bf16(O.from_bf16(S.activations_bf16(8301, len(scales), H)) * scales[:, None])
    ids = np.tile(np.arange(k, dtype=np.uint32), (len(scales), 1))
    w = np.full((len(scales), k), 0.5, np.float32)
    bufs = [nm.DeviceBuffer.from_array(a) for a in (x, ids, w)]
    out = nm.DeviceBuffer(len(scales) * H * 4)
    nm.indexed_moe_fused_decode(banks, bufs[0], nm.BF16, bufs[1], bufs[2], len(scales), k, out)
    got = out.download(np.float32).reshape(len(scales), H)
    want = O.fused_moe_decode(*stacks, O.from_bf16(x), ids, w)
    assert not got[0].any()
    for i in range(1, len(scales)):
        assert S.max_rel_err(got[i], want[i]) < TOL, scales[i]


def test_noalloc_passes_give_the_bits_of_one_pass(gpu):
    nm = gpu
    E, H, I, k, rows = 8, 512, 256, 8, 600     # 4,800 pairs: more than the fixed array holds in one pass
    banks, stacks, keep = _layer(nm, 8400, E, H, I, (Q4, Q4, Q4))
    x = S.activations_bf16(8401, rows, H)
    rng = np.random.default_rng(1)
    ids = rng.integers(0, E, (rows, k)).astype(np.uint32)
    w = rng.random((rows, k)).astype(np.float32)
    bufs = [nm.DeviceBuffer.from_array(a) for a in (x, ids, w)]
    ref, got = nm.DeviceBuffer(rows * H * 4), nm.DeviceBuffer(rows * H * 4)
    g, u, d = banks.gate.desc(), banks.up.desc(), banks.down.desc()
    for fn, out in (("naiwa_moe_decode_ex", ref), ("naiwa_moe_decode_noalloc", got)):
        rc = getattr(nm.lib(), fn)(C.byref(g), C.byref(u), C.byref(d), bufs[0].ptr, nm.BF16, bufs[1].ptr, bufs[2].ptr,
                                   rows, k, nm.ACT_SILU, out.ptr, 0, 0)
        assert rc == 0, fn
    a, b = ref.download(np.float32), got.download(np.float32)
    assert np.array_equal(a, b)
    assert S.max_rel_err(a.reshape(rows, H)[:16], O.fused_moe_decode(*stacks, O.from_bf16(x[:16]), ids[:16], w[:16])) < TOL


@pytest.mark.parametrize("dt,H,I,E,k,rows", [
    ((Q4, Q4, Q4), 256, 256, 8, 2, 5),       # 8-row tile
    ((Q4, Q4, Q8), 512, 384, 16, 3, 11),     # 16-row tile
    ((Q8, Q8, Q4), 256, 2304, 4, 2, 35),     # two K parts; chunks of 32 rows and past them
    ((Q8, Q8, Q8), 384, 128, 8, 4, 17),
])
def test_chain_rounding_at_tile_edges(gpu, dt, H, I, E, k, rows):
    """A layer of a layered step rounds x, h and the weights to bf16: within 1e-2 of the oracle,
    and the residual in the combine gives the bits of a residual launch."""
    nm = gpu
    banks, stacks, keep = _layer(nm, 8500 + rows, E, H, I, dt)
    router = S.layer(8500 + rows, E, H, I, dt)[3]
    rd = nm.DeviceBuffer.from_array(router)
    desc = (nm._lib.Layer * 1)(nm.layer_desc(rd, banks))
    x = S.activations_bf16(8501 + rows, rows, H)
    print(f"[chain {dt} H={H} I={I} E={E} k={k} rows={rows}]", flush=True)
    got = []
    for want_y in (True, False):
        xd, y = nm.DeviceBuffer.from_array(x), nm.DeviceBuffer(rows * H * 4)
        nm.stack_decode(desc, xd, rows, H, E, k, mode=O.ROUTE_SOFTMAX_TOPK_RENORM, fused=False,
                        y_out=y if want_y else None)
        nm.synchronize()
        got.append(xd.download(np.uint16))
        if want_y:
            ids, w = O.topk(O.router_logits(O.from_bf16(x), router), k, O.ROUTE_SOFTMAX_TOPK_RENORM)
            err = S.max_rel_err(y.download(np.float32).reshape(rows, H),
                                O.fused_moe_decode(*stacks, O.from_bf16(x), ids, w))
            print(f"  max_rel_err={err:.3e}", flush=True)
            assert err < 1e-2
    assert np.array_equal(got[0], got[1])


@pytest.mark.parametrize("dt,H,I,rows", [
    ((Q4, Q4, Q4), 256, 256, 4),
    ((Q4, Q4, Q8), 512, 384, 9),
    ((Q8, Q8, Q4), 384, 2304, 33),     # two K parts: the overflow in the first one
    ((Q8, Q8, Q8), 256, 256, 5),
])
def test_an_intermediate_value_past_f32_gives_infinities(gpu, dt, H, I, rows):
    """One feature of h overflows: the outputs are infinite with the sign of its down weight
    (NaN where that is zero), as a sum of products gives, and other rows are not touched."""
    nm = gpu
    rng = np.random.default_rng(rows)
    f = 5
    g, u, d = (rng.normal(0, 0.02, s).astype(np.float32) for s in ((I, H), (I, H), (H, I)))
    g[f] *= 4096
    u[f] *= 4096
    q = [O.quantize(t, a) for t, a in zip(dt, (g, u, d))]
    gw, uw, dw = (O.dequantize_f64(t, a, a0.shape[1]) for t, a, a0 in zip(dt, q, (g, u, d)))
    banks = nm.LayerBanks(1, H, I, dt)
    banks.load(0, *q)
    x = rng.normal(0, 1, (rows, H)).astype(np.float32)
    x *= np.where(x @ gw.reshape(I, H)[f].astype(np.float32) > 0, 1, -1)[:, None].astype(np.float32)  # gates of f > 0
    x[1:] *= np.float32(1e18)                         # row 0 stays ordinary
    xd = nm.DeviceBuffer.from_array(x)
    ids, w = nm.DeviceBuffer.from_array(np.zeros(rows, np.uint32)), nm.DeviceBuffer.from_array(np.ones(rows, np.float32))
    out = nm.DeviceBuffer(rows * H * 4)
    nm.indexed_moe_fused_decode(banks, xd, nm.F32, ids, w, rows, 1, out)
    got = out.download(np.float32).reshape(rows, H)
    hf = (x.astype(np.float64) @ gw.reshape(I, H)[f]) * (x.astype(np.float64) @ uw.reshape(I, H)[f])
    assert np.isfinite(got[0]).all()
    assert (np.abs(hf[1:]) > 1e39).sum() >= rows - 3
    for t in np.nonzero(np.abs(hf) > 1e39)[0]:
        want = np.sign(hf[t]) * np.sign(dw.reshape(H, I)[:, f])
        assert np.array_equal(np.isposinf(got[t]), want > 0)
        assert np.array_equal(np.isneginf(got[t]), want < 0)
        assert np.array_equal(np.isnan(got[t]), want == 0)


@pytest.mark.parametrize("dt", [(Q4, Q4, Q4), (Q8, Q8, Q8)])
@pytest.mark.parametrize("rows", [4, 12, 40])
def test_infinite_and_nan_activations_stay_in_their_rows(gpu, dt, rows):
    nm = gpu
    H = I = 512
    banks, _, keep = _layer(nm, 8600 + rows, 2, H, I, dt)
    rng = np.random.default_rng(rows)
    x = rng.normal(0, 1, (rows, H)).astype(np.float32)
    ids = nm.DeviceBuffer.from_array(rng.integers(0, 2, (rows, 2)).astype(np.uint32))
    w = nm.DeviceBuffer.from_array(np.full((rows, 2), 0.5, np.float32))

    def call(x):
        xd, out = nm.DeviceBuffer.from_array(x), nm.DeviceBuffer(rows * H * 4)
        nm.indexed_moe_fused_decode(banks, xd, nm.F32, ids, w, rows, 2, out)
        return out.download(np.float32).reshape(rows, H)

    plain = call(x)
    bad = x.copy()
    bad[1, 300] = np.inf
    bad[2, 100] = np.nan
    bad[rows - 1, 7] = -np.inf
    got = call(bad)
    assert np.isnan(got[[1, 2, rows - 1]]).all()
    others = [t for t in range(rows) if t not in (1, 2, rows - 1)]
    assert np.array_equal(got[others], plain[others])
