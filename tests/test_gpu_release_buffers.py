"""The device memory kept between shots: bounded, and given back on request
(run with -m gpu)."""
import numpy as np
import pytest

from hpcscan_amd.layout import make_layout
from tests.test_gpu_adjoint import _dev, _same

pytestmark = pytest.mark.gpu


def _shot(capi, n, nt):
    """runs one shot; (traces, bytes of its two wavefields)"""
    p = make_layout(3, n, 8)
    r = p.inner()
    at = r[0] + 3 + (r[2] + 4) * p.n1 + (r[4] + 5) * p.n1 * p.n2
    src, rec = np.array([at], np.int64), np.array([at + 2, at + p.n1], np.int64)
    g = capi.hsx_grid(p)
    coef = capi.DeviceArray(p.npoint * 4)
    capi.fill_const(g, coef, r, 0.2 * min(p.d) ** 2)
    d = [_dev(capi, x) for x in (src, np.ones((nt, 1), np.float32), rec)]
    tr = capi.DeviceArray(nt * 2 * 4)
    capi.forward(g, coef, capi.make_shot(nt, 1.0, (d[0], 1), d[1], (d[2], 2)), tr)
    return tr.download(np.float32), 2 * 4 * p.npoint


def test_kept_buffers_are_given_back(capi):
    import torch
    free = lambda: torch.cuda.mem_get_info(0)[0]
    capi.release_buffers()
    first, held = _shot(capi, (150, 140, 130), 12)
    kept = free()
    capi.release_buffers()
    given = free() - kept
    print(f"two wavefields {held} bytes, given back {given}", flush=True)
    assert given >= held
    capi.release_buffers()                     # nothing left: no effect
    assert free() - kept == given
    again, _ = _shot(capi, (150, 140, 130), 12)
    assert np.abs(first).max() > 0
    _same(again, first)
    capi.release_buffers()


def test_large_shots_keep_nothing(capi):
    """two wavefields of 310 MB: more than the library keeps"""
    import torch
    free = lambda: torch.cuda.mem_get_info(0)[0]
    _shot(capi, (420, 420, 400), 3)
    capi.release_buffers()
    before = free()
    _shot(capi, (420, 420, 400), 3)
    after = free()
    capi.release_buffers()
    assert after == before == free()
