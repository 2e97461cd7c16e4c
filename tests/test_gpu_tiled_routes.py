"""What the tests of small grids do not reach, where the library runs one thread
per point: the imaging step, gradients on the tiled kernels, every stencil with
the library's own tiles, and the pair codec of 16-bit checkpoints, each bit for
bit (run with -m gpu)."""
import ctypes

import numpy as np
import pytest

from tests.shots import make_shot
from tests.test_gpu_adjoint import _dev, _same
from tests.test_gpu_parity import PRECS, _layouts, _rand
from tests.test_gpu_row_fit import CASES as SHAPES
from tests.test_gpu_step_end import CASES as SHOTS
from tests.test_gpu_step_end import _places, _run

pytestmark = pytest.mark.gpu

_vp, _i64, _i = ctypes.c_void_p, ctypes.c_int64, ctypes.c_int


def _internal(capi, name, *argtypes):
    """a function of the library that is no entry point of its own"""
    f = getattr(capi.lib(), name)
    f.restype, f.argtypes = _i, list(argtypes)
    return f


@pytest.mark.parametrize("pair", [False, True])
@pytest.mark.parametrize("order,prec,n,lanes,rows,chunk,flags", SHAPES)
def test_imaging_step_equals_step_and_imaging(capi, oracle, order, prec, n, lanes, rows, chunk, flags, pair):
    """the fused step with the imaging condition of its output, or of its input
    and its output, against the step and the imaging conditions in turn"""
    step_img = _internal(capi, "_ZN3hsx18tiled_ac2_step_imgEPK8hsx_gridPvPKvS5_PdS5_S5_S5_S5_PKldP12ihipStream_t",
                         ctypes.POINTER(capi.HsxGrid), *[_vp] * 8, ctypes.POINTER(_i64), ctypes.c_double, _vp)
    dtype, c64 = PRECS[prec]
    p, _ = _layouts(oracle, 3, n, order, dtype)
    g = capi.hsx_grid(p, compute_fp64=c64)
    rng = np.random.default_rng(order + n[0])
    prn, prc, coef, q0, q1, q2, q3 = (_dev(capi, _rand(rng, p.npoint, dtype)) for _ in range(7))
    prn_ref = _dev(capi, prn.download(dtype))
    grad0 = _rand(rng, p.npoint, np.float64)
    grad, ref = _dev(capi, grad0), _dev(capi, grad0)
    r, scale = p.inner(), -3.7
    box = [r[0] + 1, r[1] - 1, r[2] + 1, r[3] - 1, r[4] + 1, r[5] - 1]
    print(f"imaging step order={order} {prec} n={n} rows of {p.n1} pair={pair}", flush=True)
    s = _vp()
    capi.check(capi.lib().hsx_stream_create(ctypes.byref(s)))
    capi.set_tile(lanes, chunk, rows, flags)
    try:
        capi.check(step_img(ctypes.byref(g), *(capi.dptr(x) for x in (prn, prc, coef, grad, q0, q1, q2)),
                            capi.dptr(q3) if pair else None, capi.rng(box), scale, s))
        capi.ac2_step(g, prn_ref, prc, coef, stream=s)
        if pair:
            capi.imaging(g, ref, prc, q3, q0, q1, box, scale, stream=s)
        capi.imaging(g, ref, prn_ref, q0, q1, q2, box, scale, stream=s)
        capi.sync(s)
    finally:
        capi.set_tile(0, 0)
        capi.check(capi.lib().hsx_stream_destroy(s))
    _same(prn.download(dtype), prn_ref.download(dtype))
    got, want = grad.download(np.float64), ref.download(np.float64)
    assert not np.array_equal(want, grad0)
    _same(got, want)


# small grids with a shape asked for, the large ones with the library's own
LARGE = [(8, (128, 100, 96), False), (8, (131, 101, 97), False), (4, (97, 90, 89), True)]
GRADS = [(*x, t) for x in SHOTS if x[1][0] < 100 for t in ((16, 8), (64, 16))] + [(*x, (0, 0)) for x in LARGE]


@pytest.mark.parametrize("order,n,fp64,tile", GRADS)
def test_gradient_on_the_tiled_kernels_bit_exact(oracle, capi, order, n, fp64, tile):
    """full storage and storage-type checkpoints in odd and even segments, sources
    beside the boundary planes: forward, imaging pairs and source terms"""
    print(f"tiled gradient order={order} n={n} fp64={fp64} tile={tile}", flush=True)
    sh = make_shot(oracle, n, order, nt=26, fp64=fp64, seed=order, with_obs=False)
    src, rec = _places(sh["p"], order, n)
    wav = (sh["wavelet"] * np.linspace(0.5, 1.5, len(src))).astype(sh["dtype"])
    o, coef, iv, nt = sh["o"], sh["coef"], sh["iv"], sh["nt"]
    d_obs = (0.7 * oracle.forward(o, coef, iv, nt, src, wav, rec)).astype(sh["dtype"])
    gref, _ = oracle.gradient(o, coef, iv, sh["dt"], nt, src, wav, rec, d_obs)
    assert np.abs(gref).max() > 0
    capi.set_tile(tile[0], 0, tile[1])
    try:
        for every in (0, 5, 6, 40):
            _same(_run(capi, sh, src, rec, wav, nt, every, d_obs), gref)
    finally:
        capi.set_tile(0, 0)


# arrays above the 5.2 MB from which the library takes tiles by itself, in the
# caches and (the last one, two arrays of 114 MB) not
OWN = [(order, prec, (112 + order % 3, 106, 109) if prec != "f64" else (90 + order // 2 % 2, 85, 83))
       for order in range(2, 17, 2) for prec in PRECS] + [(8, "f32", (301, 300, 290))]


@pytest.mark.parametrize("order,prec,n", OWN)
def test_own_tiles_of_every_stencil_bit_exact(oracle, capi, order, prec, n):
    dtype, c64 = PRECS[prec]
    p, o = _layouts(oracle, 3, n, order, dtype)
    assert p.npoint * np.dtype(dtype).itemsize > 5200000
    print(f"own tiles order={order} {prec} n={n} rows of {p.n1}", flush=True)
    rng = np.random.default_rng(order + n[0])
    g = capi.hsx_grid(p, compute_fp64=c64)
    u, coef, w0 = (rng.random(p.npoint, dtype=dtype) for _ in range(3))
    iv, iv1 = oracle.inv2(p.d, dtype, compute64=c64), oracle.inv1(p.d, dtype, compute64=c64)
    du, dc, dw = (_dev(capi, x) for x in (u, coef, w0))
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
    ref = w0.copy()
    oracle.pressure_fd(o, ref, u, coef, iv, compute64=c64)
    dw.upload(w0)
    capi.ac2_step(g, dw, du, dc)
    _same(dw.download(dtype), ref)


@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("fmt", ["fp16", "bf16"])
@pytest.mark.parametrize("n", [1, 3, 4, 1023, 70001])
def test_pair_codec_equals_two_snapshots(capi, fmt, n, off):
    """codes, scales and decoded values, at any length, 16-byte groups or not"""
    f = {"fp16": capi.HSX_CKPT_FP16, "bf16": capi.HSX_CKPT_BF16}[fmt]
    enc = _internal(capi, "_ZN3hsx16ckpt_encode_pairEPKfS1_lPvS2_iP12ihipStream_t", _vp, _vp, _i64, _vp, _vp, _i, _vp)
    dec = _internal(capi, "_ZN3hsx16ckpt_decode_pairEPKvS1_liPfS2_P12ihipStream_t", _vp, _vp, _i64, _i, _vp, _vp, _vp)
    rng = np.random.default_rng(n + off)
    # wavefields of neighbouring steps, zeros among them
    a = (rng.standard_normal(n + 8) * (rng.random(n + 8) < 0.9)).astype(np.float32)
    b = (a + 1e-2 * rng.standard_normal(n + 8) * (rng.random(n + 8) < 0.9)).astype(np.float32)
    da, db = _dev(capi, a), _dev(capi, b)
    at = lambda d: d.ptr.value + 4 * off
    size = capi.ckpt_bytes(n)
    blank = np.full(size, 0xAB, np.uint8)
    one, two = [_dev(capi, blank) for _ in range(2)], [_dev(capi, blank) for _ in range(2)]
    s = _vp()
    capi.check(capi.lib().hsx_stream_create(ctypes.byref(s)))
    try:
        capi.ckpt_encode(at(da), None, n, one[0], f, stream=s)
        capi.ckpt_encode(at(da), at(db), n, one[1], f, stream=s)
        capi.check(enc(at(da), at(db), n, two[0].ptr, two[1].ptr, f, s))
        capi.sync(s)
        for x, y in zip(one, two):
            assert np.array_equal(x.download(np.uint8), y.download(np.uint8))
        u1, v1, u2, v2 = (_dev(capi, np.full(n + 8, -7, np.float32)) for _ in range(4))
        capi.ckpt_decode(one[0], n, f, None, at(u1), stream=s)
        capi.ckpt_decode(one[1], n, f, at(u1), at(v1), stream=s)
        capi.check(dec(two[0].ptr, two[1].ptr, n, f, at(u2), at(v2), s))
        capi.sync(s)
        for x, y in ((u1, u2), (v1, v2)):
            assert np.array_equal(x.download(np.uint32), y.download(np.uint32))
    finally:
        capi.check(capi.lib().hsx_stream_destroy(s))
