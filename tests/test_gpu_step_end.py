"""The end of a time step in one launch with the free surface (sources and
receivers of a forward step, residual and source terms of a reverse one):
traces and gradients equal the oracle's bit for bit."""
import numpy as np
import pytest

from hpcscan_amd.layout import make_layout
from tests.shots import make_shot
from tests.test_gpu_adjoint import _dev, _same

pytestmark = pytest.mark.gpu


def _at(p, i1, i2, i3):
    r = p.inner()
    return r[0] + i1 + (r[2] + i2) * p.n1 + (r[4] + i3) * p.n1 * p.n2


def _places(p, order, n):
    """sources: two in one row (next to each end), one beside three faces, one R
    from a face; receivers: a whole row through the first two, the others, a
    scatter"""
    R = order // 2
    src = [_at(p, 1, 3, 4), _at(p, n[0] - 2, 3, 4), _at(p, 2, n[1] - 2, 1), _at(p, n[0] // 2, R, n[2] - 1 - R)]
    rec = [_at(p, i, 3, 4) for i in range(1, n[0] - 1)] + src[2:] + [_at(p, 1 + k % 3, 1 + k, 2) for k in range(n[1] - 2)]
    return np.unique(src).astype(np.int64), np.unique(rec).astype(np.int64)


def _run(capi, sh, src, rec, wav, nt, every=None, d_obs=None):
    g = capi.hsx_grid(sh["p"])
    dsrc, drec, dwav, dcoef = (_dev(capi, x) for x in (src, rec, wav, sh["coef"]))
    s = capi.make_shot(nt, sh["dt"], (dsrc, len(src)), dwav, (drec, len(rec)))
    if every is None:
        tr = capi.DeviceArray(nt * len(rec) * np.dtype(sh["dtype"]).itemsize)
        capi.forward(g, dcoef, s, tr)
        return tr.download(sh["dtype"]).reshape(nt, len(rec))
    grad = _dev(capi, np.zeros(sh["p"].npoint))
    capi.gradient(g, dcoef, s, _dev(capi, d_obs), grad, every, capi.HSX_CKPT_FP32)
    return grad.download(np.float64)


# the smallest grid of the one-launch free surface (R + 2 points) of order 16,
# rows of odd length and whole vectors, a grid of the tiled kernels
CASES = [(8, (61, 20, 18), False), (8, (24, 20, 18), True), (4, (23, 12, 11), False), (2, (16, 9, 8), False),
         (6, (21, 13, 12), True), (16, (12, 11, 10), False), (8, (128, 100, 96), False)]


@pytest.mark.parametrize("order,n,fp64", CASES)
def test_step_end_bit_exact(oracle, capi, order, n, fp64):
    print(f"step end order={order} n={n} fp64={fp64}", flush=True)
    big = n[0] > 100
    sh = make_shot(oracle, n, order, nt=26, fp64=fp64, seed=order, with_obs=False)
    src, rec = _places(sh["p"], order, n)
    wav = (sh["wavelet"] * np.linspace(0.5, 1.5, len(src))).astype(sh["dtype"])
    o, coef, iv, nt = sh["o"], sh["coef"], sh["iv"], sh["nt"]
    ref = oracle.forward(o, coef, iv, nt, src, wav, rec)
    assert np.abs(ref).max() > 0
    _same(_run(capi, sh, src, rec, wav, nt), ref)
    # receivers on the n2 and n3 planes (one of them twice) stay with the one
    # launch; one on the n1 plane, or too many, takes the separate launches
    p = sh["p"]
    m2, m3 = n[1] - 1, n[2] - 1
    edge = [_at(p, *x) for x in ((1, 0, 4), (n[0] - 2, m2, 4), (3, 3, 0), (1, 1, m3), (n[0] // 2, 0, 0), (2, m2, m3))]
    for more in (edge + edge[:1], edge + [_at(p, 0, 4, 4)], [_at(p, i, 0, 2) for i in range(1, n[0] - 1)] + edge * 3):
        rec2 = np.concatenate([rec, more]).astype(np.int64)
        _same(_run(capi, sh, src, rec2, wav, nt), oracle.forward(o, coef, iv, nt, src, wav, rec2))
    if big:
        return
    d_obs = (0.7 * ref).astype(sh["dtype"])
    gref, _ = oracle.gradient(o, coef, iv, sh["dt"], nt, src, wav, rec, d_obs)
    assert np.abs(gref).max() > 0
    for every in (0, 1, 2, 5, 40):
        _same(_run(capi, sh, src, rec, wav, nt, every, d_obs), gref)


@pytest.mark.parametrize("every", [1, 6, 40])
def test_16bit_segments(oracle, capi, every):
    """16-bit checkpoints of every step, of odd and even segments, of one segment"""
    sh = make_shot(oracle, (24, 20, 18), 8, nt=45, seed=11)
    src, rec = sh["src"], sh["rec"]
    gref, _ = oracle.gradient(sh["o"], sh["coef"], sh["iv"], sh["dt"], sh["nt"], src, sh["wavelet"], rec, sh["d_obs"])
    g = capi.hsx_grid(sh["p"])
    dsrc, drec, dwav, dcoef = (_dev(capi, x) for x in (src, rec, sh["wavelet"], sh["coef"]))
    s = capi.make_shot(sh["nt"], sh["dt"], (dsrc, len(src)), dwav, (drec, len(rec)))
    grad = _dev(capi, np.zeros(sh["p"].npoint))
    capi.gradient(g, dcoef, s, _dev(capi, sh["d_obs"]), grad, every, capi.HSX_CKPT_FP16)
    # the bound of the 16-bit checkpoints' own test; a segment is redone from its start
    assert np.linalg.norm(grad.download(np.float64) - gref) < 1e-3 * np.linalg.norm(gref)


def test_two_dimensions(capi):
    """the first 20 of 30 steps (one launch) equal a run of 20 (separate launches)"""
    p = make_layout(2, (65, 41), 8)
    coef = np.zeros(p.npoint, np.float32)
    r = p.inner()
    c = coef.reshape(p.n2, p.n1)
    c[r[2]:r[3] + 1, r[0]:r[1] + 1] = np.float32(0.2 * min(p.d[:2]) ** 2)
    sh = {"p": p, "coef": coef, "dt": 1.0, "dtype": np.float32}
    src = np.array([r[0] + 1 + (r[2] + 2) * p.n1, r[1] - 2 + (r[2] + 2) * p.n1], np.int64)
    rec = np.array([r[0] + k + (r[2] + 2) * p.n1 for k in range(1, 64)], np.int64)
    wav = np.random.default_rng(3).standard_normal((30, 2)).astype(np.float32)
    a, b = _run(capi, sh, src, rec, wav, 30), _run(capi, sh, src, rec, wav[:20], 20)
    assert np.abs(b).max() > 0
    _same(a[:20], b)


def test_shots_on_two_threads(oracle, capi):
    """shots of different sizes on two threads and streams, whose buffers serve
    one call after another: each one's traces stay its own"""
    import threading

    import torch
    jobs = []
    for k, n in enumerate([(24, 20, 18), (61, 20, 18), (30, 25, 22), (24, 20, 18)]):
        sh = make_shot(oracle, n, 8, nt=30, seed=40 + k, with_obs=False)
        d = [_dev(capi, sh[x]) for x in ("src", "rec", "wavelet", "coef")]
        tr = capi.DeviceArray(30 * len(sh["rec"]) * 4)
        desc = capi.make_shot(30, sh["dt"], (d[0], len(sh["src"])), d[2], (d[1], len(sh["rec"])))
        ref = oracle.forward(sh["o"], sh["coef"], sh["iv"], 30, sh["src"], sh["wavelet"], sh["rec"])
        jobs.append((capi.hsx_grid(sh["p"]), d[3], desc, tr, ref, d))
    streams = [torch.cuda.Stream() for _ in range(2)]

    def work(i):
        for _ in range(5):
            for g, coef, desc, tr, _, _ in jobs[i::2]:
                capi.forward(g, coef, desc, tr, stream=streams[i].cuda_stream)

    ts = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for _, _, _, tr, ref, _ in jobs:
        _same(tr.download(np.float32).reshape(ref.shape), ref)
