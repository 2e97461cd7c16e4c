"""Receivers (and sources) outside the inner points: in the halos, in their
corners, beyond them.  A shot whose steps are out of place (full storage,
storage-type checkpoints) records what one whose steps are in place does:
misfit and gradient equal the oracle's, also on a plan whose buffers hold
another gradient's wavefields (run with -m gpu)."""
import numpy as np
import pytest

from tests.shots import make_shot
from tests.test_gpu_adjoint import _dev, _same

pytestmark = pytest.mark.gpu


# nt below and above the least for the merged step ends; sources in one launch
# with the receivers (1 and 3) and in one of their own (70), some of them outside
@pytest.mark.parametrize("fp64,nt,nsrc", [(False, 12, 1), (False, 30, 3), (True, 30, 3), (False, 30, 70), (True, 9, 70)])
@pytest.mark.parametrize("every", [0, 2, 5, 40])
def test_receivers_outside_the_inner_points(oracle, capi, fp64, nt, nsrc, every):
    print(f"outside receivers fp64={fp64} nt={nt} nsrc={nsrc} every={every}", flush=True)
    sh = make_shot(oracle, (20, 18, 16), 8, nt=nt, fp64=fp64, seed=7, with_obs=False)
    p, r = sh["p"], sh["p"].inner()
    at = lambda i1, i2, i3: i1 + i2 * p.n1 + i3 * p.n1 * p.n2
    c1, c2, c3 = r[0] + 2, (r[2] + r[3]) // 2, (r[4] + r[5]) // 2
    # halos of each face, corners, the planes, inner points
    rec = np.array([at(r[0] - 2, c2, c3), at(r[1] + 1, c2, c3), at(c1, r[2] - 2, c3), at(c1, r[3] + 3, c3),
                    at(c1, c2, r[4] - 1), at(c1, c2, r[5] + 4), at(r[0] - 2, c2 + 1, c3), at(0, 0, 0), at(r[0] - 1, r[2] - 1, c3),
                    at(p.n1 - 1, p.n2 - 1, p.n3 - 1), at(r[0], c2, c3), at(c1, c2 + 1, c3), at(c1 + 1, c2, c3)], np.int64)
    rng = np.random.default_rng(nsrc)
    inner = np.flatnonzero(sh["inner_mask"])
    # the shot's own source; a corner and a halo point that are receivers; inner points
    src = np.concatenate([sh["src"], [at(0, 0, 0), at(r[0] - 2, c2, c3)][:nsrc - 1],
                          rng.choice(inner[~np.isin(inner, sh["src"])], max(0, nsrc - 3), replace=False)]).astype(np.int64)
    assert len(src) == nsrc
    wav = (np.repeat(sh["wavelet"], nsrc, axis=1) + rng.uniform(-1e-3, 1e-3, (nt, nsrc))).astype(sh["dtype"])
    o, coef, iv = sh["o"], sh["coef"], sh["iv"]
    g = capi.hsx_grid(p)
    dsrc, drec, dcoef = (_dev(capi, x) for x in (src, rec, coef))
    plan = capi.AdjointPlan(g, nt, len(rec), every, capi.HSX_CKPT_FP32)
    for amp in (1e3, 1.0):                     # the second gradient finds the first one's wavefields
        w = (amp * wav).astype(sh["dtype"])
        ref = oracle.forward(o, coef, iv, nt, src, w, rec)
        assert np.abs(ref[:, :8]).max() > 0
        d_obs = (0.7 * ref).astype(sh["dtype"])
        gref, jref = oracle.gradient(o, coef, iv, sh["dt"], nt, src, w, rec, d_obs)
        dw = _dev(capi, w)
        s = capi.make_shot(nt, sh["dt"], (dsrc, nsrc), dw, (drec, len(rec)))
        grad = _dev(capi, np.zeros(p.npoint))
        j = plan.gradient(g, dcoef, s, _dev(capi, d_obs), grad)
        assert j == pytest.approx(jref, rel=1e-12)
        _same(grad.download(np.float64), gref)
        tr = capi.DeviceArray(nt * len(rec) * np.dtype(sh["dtype"]).itemsize)
        capi.forward(g, dcoef, s, tr)
        _same(tr.download(sh["dtype"]).reshape(ref.shape), ref)
    plan.close()
