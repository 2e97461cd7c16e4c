"""The device memory kept between shots: bounded, and given back on request
(run with -m gpu)."""
import time

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


def _free(at_least=None):
    """bytes free on the device; the driver clears freed memory before it counts
    as free, so what has to come back is waited for (10 s at most)"""
    import torch
    for _ in range(200):
        now = torch.cuda.mem_get_info(0)[0]
        if at_least is None or now >= at_least:
            break
        time.sleep(0.05)
    return now


PAGE = 2 << 20                                 # device memory is handed out and counted in these


def test_kept_buffers_are_given_back(capi):
    capi.release_buffers()
    first, held = _shot(capi, (300, 280, 260), 12)
    time.sleep(1)                              # what the shot itself freed
    kept = _free()
    capi.release_buffers()
    # whole pages inside the buffer; its first and last may hold something else too
    pages = held // PAGE - 1
    given = _free(kept + pages * PAGE) - kept
    print(f"two wavefields {held} bytes, given back {given}", flush=True)
    assert given >= pages * PAGE
    capi.release_buffers()                     # nothing left: no effect
    again, _ = _shot(capi, (300, 280, 260), 12)
    assert np.abs(first).max() > 0
    _same(again, first)
    capi.release_buffers()


def test_large_shots_keep_nothing(capi):
    """two wavefields of 310 MB: more than the library keeps"""
    _shot(capi, (420, 420, 400), 3)
    capi.release_buffers()
    time.sleep(1)
    before = _free()
    _shot(capi, (420, 420, 400), 3)
    assert _free(before) >= before
