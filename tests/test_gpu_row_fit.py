"""Tiles fitted to the row: rows that are not whole 16-byte vectors (odd sizes
and halo widths, tiles that start before the first point), and tile widths that
are no power of two, bit for bit against the oracle (run with -m gpu)."""
import numpy as np
import pytest

from test_gpu_parity import PRECS, _layouts, _rand, _same

pytestmark = pytest.mark.gpu

CASES = [
    # (order, prec, n, lanes, rows, chunk, flags); n1 = n[0] + order (+ 1 where the halo is odd, FP32)
    (2, "f32", (100, 20, 22), 64, 16, 0, 0),      # inner start 2, tiles from -1: rows read from the row before
    (2, "f32", (6, 9, 7), 16, 8, 3, 0),           # rows of nine points
    (2, "f32", (101, 17, 19), 32, 8, 4, 0),       # whole vectors from 0
    (2, "f64", (31, 12, 9), 16, 8, 0, 0),         # FP64, tiles from 0 or 1
    (4, "f32", (403, 37, 25), 128, 8, 0, 0),      # 101 lanes of 128
    (4, "f32", (201, 18, 23), 64, 16, 0, 4),      # 51 lanes, no ring
    (6, "f32", (250, 33, 21), 64, 16, 0, 0),      # R = 3, ring, 63 lanes kept at 64
    (6, "f32c64", (77, 21, 18), 32, 8, 5, 0),
    (8, "f32", (200, 40, 30), 64, 8, 6, 4),       # 50 lanes, aligned rows
    (8, "f32", (300, 21, 30), 64, 16, 0, 0),      # two tiles of 40 lanes
    (8, "f32", (303, 21, 30), 64, 16, 7, 0),      # the same with rows at any address
    (8, "f32", (610, 12, 20), 128, 8, 0, 0),      # two tiles of 80 lanes
    (8, "f64", (99, 23, 20), 32, 16, 0, 0),
    (10, "f32", (129, 24, 27), 32, 8, 0, 0),      # R = 5
    (12, "f64", (61, 26, 30), 64, 8, 9, 0),
    (14, "f32", (119, 31, 33), 32, 16, 0, 0),     # R = 7
    (16, "f32", (33, 35, 37), 16, 8, 0, 0),       # 9 lanes
    (16, "f64", (35, 34, 33), 16, 8, 0, 0),       # four halo columns per side
]


@pytest.mark.parametrize("order,prec,n,lanes,rows,chunk,flags", CASES)
def test_rows_of_any_length_bit_exact(oracle, capi, order, prec, n, lanes, rows, chunk, flags):
    dtype, c64 = PRECS[prec]
    p, o = _layouts(oracle, 3, n, order, dtype)
    rng = np.random.default_rng(order * 13 + n[0])
    g = capi.hsx_grid(p, compute_fp64=c64)
    u, coef, prn, w0 = (_rand(rng, p.npoint, dtype) for _ in range(4))
    iv, iv1 = oracle.inv2(p.d, dtype, compute64=c64), oracle.inv1(p.d, dtype, compute64=c64)
    du, dc, dp, dw = (capi.DeviceArray.from_numpy(x) for x in (u, coef, prn, w0))
    print(f"order={order} prec={prec} n={n} rows of {p.n1}", flush=True)
    capi.set_tile(lanes, chunk, rows, flags)      # a shape asked for is used on any rows
    try:
        for axis in range(3):
            for op, ref_op, x in ((capi.fd_d2, oracle.fd_d2, iv), (capi.fd_d1, oracle.fd_d1, iv1)):
                ref = w0.copy()
                ref_op(o, axis, u, ref, x, compute64=c64)
                dw.upload(w0)
                op(g, axis, du, dw)
                _same(dw.download(dtype), ref)
        ref = w0.copy()
        oracle.laplacian(o, u, ref, iv, compute64=c64)
        dw.upload(w0)
        capi.laplacian(g, du, dw)
        _same(dw.download(dtype), ref)
        ref = prn.copy()
        oracle.pressure_fd(o, ref, u, coef, iv, compute64=c64)
        capi.ac2_step(g, dp, du, dc)
        _same(dp.download(dtype), ref)
    finally:
        capi.set_tile(0, 0)


# one grid of each class of the library's own shapes (5 MB an array, 200 MB for
# the step's three, above by precision and order), no shape asked for
CLASSES = [(8, "f32", (90, 85, 80)), (8, "f32", (160, 150, 141)), (12, "f32", (161, 120, 130)),
           (8, "f64", (130, 100, 90)), (8, "f32c64", (150, 141, 100)), (8, "f32", (300, 280, 270)),
           (4, "f32", (301, 280, 270)), (16, "f32", (300, 260, 240)), (8, "f64", (260, 240, 200)),
           (12, "f32c64", (300, 250, 240)), (8, "f32c64", (300, 260, 250)), (4, "f32c64", (400, 330, 300))]


@pytest.mark.parametrize("order,prec,n", CLASSES)
def test_own_shapes_bit_exact(oracle, capi, order, prec, n):
    dtype, c64 = PRECS[prec]
    p, o = _layouts(oracle, 3, n, order, dtype)
    rng = np.random.default_rng(order + n[0])
    g = capi.hsx_grid(p, compute_fp64=c64)
    u, coef, prn = (rng.random(p.npoint, dtype=dtype) for _ in range(3))
    iv = oracle.inv2(p.d, dtype, compute64=c64)
    du, dc, dp = (capi.DeviceArray.from_numpy(x) for x in (u, coef, prn))
    ref = prn.copy()
    oracle.pressure_fd(o, ref, u, coef, iv, compute64=c64)
    capi.ac2_step(g, dp, du, dc)
    _same(dp.download(dtype), ref)
    ref = prn.copy()
    oracle.laplacian(o, u, ref, iv, compute64=c64)
    dp.upload(prn)
    capi.laplacian(g, du, dp)
    _same(dp.download(dtype), ref)
