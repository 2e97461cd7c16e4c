"""The 16-bit snapshots in vectors: codes and values at any alignment and length."""
import numpy as np
import pytest

from tests.test_gpu_adjoint import _dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt", ["fp16", "bf16"])
@pytest.mark.parametrize("n", [1, 3, 4, 1023, 70001])
def test_codec_any_alignment(capi, fmt, n):
    """16-byte groups, their tail, and buffers at any element address: the same codes and values"""
    f = {"fp16": capi.HSX_CKPT_FP16, "bf16": capi.HSX_CKPT_BF16}[fmt]
    rng = np.random.default_rng(n)
    u, v = (rng.standard_normal(n + 4).astype(np.float32) for _ in range(2))
    got = []
    for off in (0, 1):
        pad = lambda x: _dev(capi, np.concatenate([np.zeros(off, np.float32), x[:n], np.zeros(8, np.float32)]))
        du, dv, out = pad(u), pad(v), pad(np.zeros(n + 4, np.float32))
        at = lambda d: d.ptr.value + 4 * off
        packed = capi.DeviceArray(capi.ckpt_bytes(n))
        for prev in (None, at(dv)):
            capi.ckpt_encode(at(du), prev, n, packed, f)
            capi.ckpt_decode(packed, n, f, at(du) if prev else None, at(out))
            got.append((off, prev is not None, packed.download(np.uint8)[:256 + 2 * n].copy(),
                        out.download(np.float32)[off:off + n].copy()))
    for k in range(2):
        a, b = got[k], got[k + 2]
        assert np.array_equal(a[2][:8], b[2][:8]) and np.array_equal(a[2][256:], b[2][256:])
        assert np.array_equal(a[3], b[3])
        # rounded to 11 (8) bits relative to the value, and to the format's smallest step
        want = (u if k == 0 else v)[:n]
        scale = np.abs(u[:n] if k == 0 else u[:n] - v[:n]).max()
        assert np.abs(a[3] - want).max() <= scale * (2.0 ** -11 if fmt == "fp16" else 2.0 ** -8) * 1.01
