"""Free surface in one launch, and the 2D step and Laplacian in vectors, bit
for bit against the oracle (run with -m gpu)."""
import numpy as np
import pytest

from test_gpu_parity import PRECS, _layouts, _rand, _same

pytestmark = pytest.mark.gpu

# (order, prec, n): rows of whole vectors and not, the smallest axes the closed
# form takes (R + 2 points: every inner point mirrors into both halos), 1D-3D
SURFACES = [
    (2, "f32", (3, 3, 3)), (2, "f32", (37,)), (2, "f64", (5, 4, 6)), (4, "f32", (4, 4, 4)), (4, "f32", (23, 19)),
    (6, "f32", (17, 6, 9)), (8, "f32", (6, 6, 6)), (8, "f32", (20, 21, 7)), (8, "f32", (21, 18, 17)),
    (8, "f32", (131, 70)), (8, "f64", (19, 6, 8)), (12, "f32", (40, 9, 8)), (12, "f64", (26, 11, 10)),
    (14, "f32", (33, 9, 12)), (16, "f32", (32, 10, 30)), (16, "f64", (31, 12, 10)),
]


@pytest.mark.parametrize("order,prec,n", SURFACES)
def test_free_surface_every_mask_bit_exact(oracle, capi, order, prec, n):
    """Whole grids, signs of zero included, for every mask of faces."""
    dtype, c64 = PRECS[prec]
    p, o = _layouts(oracle, len(n), n, order, dtype)
    g = capi.hsx_grid(p, compute_fp64=c64)
    u = _rand(np.random.default_rng(order + n[0]), p.npoint, dtype)
    d = capi.DeviceArray.from_numpy(u)
    for mask in range(1, 1 << (2 * len(n))):
        ref = u.copy()
        oracle.free_surface(o, ref, compute64=c64, face_mask=mask)
        d.upload(u)
        capi.free_surface(g, d, face_mask=mask)
        assert np.array_equal(d.download(dtype).view(np.uint8), ref.view(np.uint8)), f"mask {mask:#x}"


# (order, prec, n): rows that start before the first point (order 2 FP32), a
# last vector that ends at the row's end; two rows per lane from 1500 waves of
# vectors on, four from 8192, one thread per point below
PLANES = [(2, "f32", (100, 9)), (2, "f32", (100, 4003)), (2, "f32", (7, 50021)), (2, "f64", (33, 8200)),
          (4, "f32", (6, 300007)), (4, "f32", (257, 50)),
          (6, "f32", (301, 2101)), (8, "f32", (1003, 2099)), (8, "f32", (64, 64)), (8, "f32", (1501, 1030)), (8, "f64", (203, 41)),
          (8, "f32c64", (130, 2051)), (10, "f32", (99, 33)), (12, "f64", (129, 4097)), (16, "f32", (515, 2049)),
          (16, "f64", (65, 23)), (16, "f32c64", (18, 4099))]


@pytest.mark.parametrize("order,prec,n", PLANES)
def test_2d_step_and_laplacian_bit_exact(oracle, capi, order, prec, n):
    dtype, c64 = PRECS[prec]
    p, o = _layouts(oracle, 2, n, order, dtype)
    rng = np.random.default_rng(order * 5 + n[0])
    g = capi.hsx_grid(p, compute_fp64=c64)
    u, coef, prn, w0 = (_rand(rng, p.npoint, dtype) for _ in range(4))
    iv = oracle.inv2(p.d, dtype, compute64=c64)
    du, dc, dp, dw, do = (capi.DeviceArray.from_numpy(x) for x in (u, coef, prn, w0, w0))
    ref = w0.copy()
    oracle.laplacian(o, u, ref, iv, compute64=c64)
    capi.laplacian(g, du, dw)
    _same(dw.download(dtype), ref)
    ref = prn.copy()
    oracle.pressure_fd(o, ref, u, coef, iv, compute64=c64)
    capi.ac2_step_to(g, do, dp, du, dc)           # out of place: prn is left alone
    _same(dp.download(dtype), prn)
    inner = np.zeros((p.n2, p.n1), bool)
    r = p.inner()
    inner[r[2]:r[3] + 1, r[0]:r[1] + 1] = True
    _same(do.download(dtype), np.where(inner.ravel(), ref, w0))
    capi.ac2_step(g, dp, du, dc)
    _same(dp.download(dtype), ref)
