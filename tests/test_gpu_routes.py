"""Which kernel a call runs: shapes asked for, tuned shapes, grids at the ends of
the rules (run with -m gpu)."""
import numpy as np
import pytest

from hpcscan_amd.layout import make_layout
from tests.launches import launches
from tests.shots import make_shot
from tests.test_gpu_adjoint import _dev, _same, _shot_dev
from tests.test_gpu_parity import PRECS, _layouts, _rand

pytestmark = pytest.mark.gpu


def _step(capi, p, **kw):
    """the launches of the fused step on zero grids of p"""
    g = capi.hsx_grid(p, **kw)
    prn, prc, coef = (capi.DeviceArray(p.npoint * (8 if p.fp64 else 4)) for _ in range(3))
    for d in (prn, prc, coef):
        capi.array_op(g, capi.HSX_ARRAY_FILL, d, val=0.0)
    capi.sync()
    return launches(capi, lambda s: capi.ac2_step(g, prn, prc, coef, stream=s))


# below the tiled kernels' own range (the tuner keeps one thread per point or a
# tile shape, whichever is faster) and in it
TUNED = [((100, 100, 100), 8, "f32"), ((40, 36, 32), 8, "f32"), ((60, 60, 60), 8, "f32"), ((128, 120, 110), 8, "f32"),
         ((80, 70, 70), 8, "f64"), ((40, 36, 32), 8, "f64"), ((72, 62, 62), 16, "f64"), ((32, 32, 32), 16, "f64"),
         ((96, 90, 90), 8, "f32c64"), ((88, 80, 80), 16, "f32c64"), ((88, 90, 80), 16, "f32"), ((32, 32, 32), 16, "f32")]


@pytest.mark.parametrize("n,order,prec", TUNED)
def test_step_runs_what_the_tuner_reports(capi, n, order, prec):
    """the step on a tuned grid runs the shape that hsx_autotune returned, the
    one that its time is of; 0, 0, 0, 0 is what the step runs untuned"""
    p = make_layout(3, n, order, fp64=prec == "f64")
    kw = {"compute_fp64": prec != "f32"}
    capi.autotune_clear()
    try:
        own = _step(capi, p, **kw)
        shape, ms = capi.autotune(capi.hsx_grid(p, **kw), reps=20)
        print(f"n={n} order={order} {prec}: own {own}, tuned {shape} {1e3 * ms:.2f} us", flush=True)
        tuned = _step(capi, p, **kw)
        capi.autotune_clear()
        lanes, rows, chunk, flags = shape
        capi.set_tile(lanes, chunk, rows, flags)
        assert tuned == _step(capi, p, **kw)
    finally:
        capi.set_tile(0, 0)
        capi.autotune_clear()
    assert _step(capi, p, **kw) == own


def test_tuned_time_is_the_steps(capi):
    """32 points an axis, order 16: a launch of any tile shape lasts three times
    as long as one thread per point; the tuner's time is that of the step"""
    import ctypes
    p = make_layout(3, (32, 32, 32), 16)
    g = capi.hsx_grid(p)
    prn, prc, coef = (_dev(capi, np.zeros(p.npoint, np.float32)) for _ in range(3))
    stream, e0, e1, ms = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_float()
    L = capi.lib()
    capi.check(L.hsx_stream_create(ctypes.byref(stream)))
    for e in (e0, e1):
        capi.check(L.hsx_event_create(ctypes.byref(e)))
    capi.autotune_clear()
    try:
        told = min(capi.autotune(g, reps=50)[1] for _ in range(3))
        ran = []
        for _ in range(5):
            capi.ac2_step(g, prn, prc, coef, stream=stream)
            capi.check(L.hsx_event_record(e0, stream))
            for _ in range(50):
                capi.ac2_step(g, prn, prc, coef, stream=stream)
            capi.check(L.hsx_event_record(e1, stream))
            capi.sync(stream)
            capi.check(L.hsx_event_elapsed_ms(e0, e1, ctypes.byref(ms)))
            ran.append(ms.value / 50)
    finally:
        capi.autotune_clear()
        for e in (e0, e1):
            capi.check(L.hsx_event_destroy(e))
        capi.check(L.hsx_stream_destroy(stream))
    print(f"tuner {1e3 * told:.2f} us, step {1e3 * min(ran):.2f} us", flush=True)
    # (the step may be bound by this loop's launches)
    assert told < 2 * min(ran)


def test_plan_with_a_tuned_shape_bit_exact(oracle, capi):
    """a plan made with HSX_ADJ_AUTOTUNE on a grid below the tiled kernels' own
    range, whose forward and reverse steps run the tuned shape"""
    sh = make_shot(oracle, (72, 62, 62), 16, nt=25, fp64=True, seed=38)
    g = capi.hsx_grid(sh["p"])
    d, s = _shot_dev(capi, sh)
    capi.autotune_clear()
    try:
        plan = capi.AdjointPlan(g, sh["nt"], len(sh["rec"]), 6, capi.HSX_CKPT_FP32, autotune=True)
        grad = _dev(capi, np.zeros(sh["p"].npoint))
        plan.gradient(g, d["coef"], s, _dev(capi, sh["d_obs"]), grad)
        plan.close()
    finally:
        capi.autotune_clear()
    gref, _ = oracle.gradient(sh["o"], sh["coef"], sh["iv"], sh["dt"], sh["nt"], sh["src"], sh["wavelet"],
                              sh["rec"], sh["d_obs"])
    assert np.abs(gref).max() > 0
    _same(grad.download(np.float64), gref)


@pytest.mark.parametrize("n3", [65535, 65536, 70000])
def test_more_planes_than_one_launch_of_points(oracle, capi, n3):
    """a small array (4.5 MB) of more than 65535 planes, which only the tiled
    kernels take: step, Laplacian, D2 and D1 equal the oracle's"""
    dtype, c64 = PRECS["f32"]
    p, o = _layouts(oracle, 3, (2, 2, n3), 2, dtype, offset=(0, 0, 0))
    assert p.n1 == p.n2 == 4
    rng = np.random.default_rng(n3)
    g = capi.hsx_grid(p, compute_fp64=c64)
    u, coef, prn, w0 = (_rand(rng, p.npoint, dtype) for _ in range(4))
    iv, iv1 = oracle.inv2(p.d, dtype, compute64=c64), oracle.inv1(p.d, dtype, compute64=c64)
    du, dc, dp, dw = (_dev(capi, x) for x in (u, coef, prn, w0))
    ref = prn.copy()
    oracle.pressure_fd(o, ref, u, coef, iv, compute64=c64)
    capi.ac2_step(g, dp, du, dc)
    _same(dp.download(dtype), ref)
    ref = w0.copy()
    oracle.laplacian(o, u, ref, iv, compute64=c64)
    capi.laplacian(g, du, dw)
    _same(dw.download(dtype), ref)
    for axis in range(3):
        for op, ref_op, x in ((capi.fd_d2, oracle.fd_d2, iv), (capi.fd_d1, oracle.fd_d1, iv1)):
            ref = w0.copy()
            ref_op(o, axis, u, ref, x, compute64=c64)
            dw.upload(w0)
            op(g, axis, du, dw)
            _same(dw.download(dtype), ref)


# one grid of each of the step's own tiles: 128 x 8 with the ring, 64 x 8 in the
# caches, 32 x 16 FP64, 32 x 8 with 12-plane chunks
@pytest.mark.parametrize("n,order,prec,flags", [((508, 270, 130), 8, "f32", 1), ((128, 120, 110), 8, "f32", 6),
                                                ((260, 240, 200), 8, "f64", 6), ((280, 260, 250), 8, "f32c64", 6)])
def test_a_partly_given_shape_keeps_the_own_tile(capi, n, order, prec, flags):
    """only a chunk or only flags asked for: lanes, rows and what else is left 0
    stay the library's choice, and results the same"""
    p = make_layout(3, n, order, fp64=prec == "f64")
    kw = {"compute_fp64": prec != "f32"}
    g = capi.hsx_grid(p, **kw)
    rng = np.random.default_rng(5)
    u, coef, prn = (rng.random(p.npoint, dtype=p.dtype) for _ in range(3))
    du, dc, dp = (_dev(capi, x) for x in (u, coef, prn))
    got = []
    try:
        for chunk, fl in ((0, 0), (20, 0), (0, flags)):
            capi.set_tile(0, chunk, 0, fl)
            (run,) = _step(capi, p, **kw)
            dp.upload(prn)
            capi.ac2_step(g, dp, du, dc)
            got.append((run, dp.download(p.dtype)))
            print(f"n={n} {prec} chunk {chunk} flags {fl}: {run}", flush=True)
    finally:
        capi.set_tile(0, 0)
    own, chunked, flagged = (x[0] for x in got)
    assert chunked[1:] == own[1:]              # threads and LDS bytes of the tile
    assert flagged == own                      # flags: the own choice of the ring, other streams
    for x in got[1:]:
        _same(x[1], got[0][1])


# rows of few lanes, whose workgroups have 72 to 256 threads
NARROW = [((64, 300, 200), 8, "f32"), ((61, 61, 700), 4, "f32"), ((40, 300, 300), 8, "f32"), ((64, 400, 100), 6, "f32c64"),
          ((250, 120, 200), 12, "f32c64"), ((200, 190, 180), 12, "f32")]


@pytest.mark.parametrize("n,order,prec", NARROW)
def test_narrow_tiles_fill_the_chip(capi, n, order, prec):
    """grids in the caches: two workgroups per CU are a full launch only where a
    workgroup has 400 threads or more; smaller ones come in larger numbers"""
    p = make_layout(3, n, order)
    g = capi.hsx_grid(p, compute_fp64=prec == "f32c64")
    cus = capi.device_info(0)["compute_units"]
    a, b, c = (capi.DeviceArray(p.npoint * 4) for _ in range(3))
    for d in (a, b, c):
        capi.array_op(g, capi.HSX_ARRAY_FILL, d, val=0.0)
    capi.sync()
    for op in (lambda s: capi.ac2_step(g, a, b, c, stream=s), lambda s: capi.laplacian(g, b, a, stream=s),
               lambda s: capi.fd_d2(g, 0, b, a, stream=s), lambda s: capi.fd_d1(g, 1, b, a, stream=s)):
        ((grid, block, lds),) = launches(capi, op)
        print(f"n={n} order={order} {prec}: {grid[0]} workgroups of {block[0]}", flush=True)
        assert block[1] == 1 and block[0] <= 512         # a tile of the cached shape
        assert block[0] >= 400 or grid[0] > 2 * cus


@pytest.mark.parametrize("fp64", [False, True])
def test_n1_faces_alone_keep_their_kernel(capi, fp64):
    """faces along n1 only, rows of whole vectors: the kernel of the row ends, one
    launch; with other faces the one that leaves their rows out"""
    p = make_layout(3, (60, 50, 40), 8, fp64=fp64)
    g = capi.hsx_grid(p)
    u = _dev(capi, np.zeros(p.npoint, p.dtype))
    run = {m: launches(capi, lambda s: capi.free_surface(g, u, face_mask=m, stream=s), func=True) for m in (1, 3, 7, 63)}
    assert all(len(x) == 1 for x in run.values())
    kernel = {m: x[0][3] for m, x in run.items()}
    assert kernel[1] == kernel[3] != kernel[7] == kernel[63]
