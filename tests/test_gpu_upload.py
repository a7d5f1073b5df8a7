"""Uploads around the size that travels in a kernel's arguments (1 KiB), from
either host type: the values, their order with later work, and that the host
buffer may change as soon as the call returns."""
import ctypes

import numpy as np
import pytest

from picoquant_hip import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("host", [np.complex128, np.complex64])
@pytest.mark.parametrize("n", [1, 2, 16, 63, 64, 65, 128, 129, 1000])
def test_upload_sizes(dtype, host, n):
    ctx = _lib.Context(dtype)
    try:
        rng = np.random.default_rng(n)
        hs, want = [], []
        buf = np.empty(n, dtype=host)
        for _ in range(20):
            buf[:] = rng.standard_normal(n) + 1j * rng.standard_normal(n)
            want.append(buf.astype(dtype))
            hs.append(ctx.upload(buf))
            buf[:] = 0
        # a contraction right behind its operands' uploads
        hc = ctx.contract(hs[-1], [1], hs[-2], [1])
        got = complex(ctx.download(hc))
        ref = np.sum(want[-1].astype(np.complex128) * want[-2].astype(np.complex128))
        scale = np.sum(np.abs(want[-1]) * np.abs(want[-2]))
        assert abs(got - ref) <= (1e-12 if dtype == np.complex128 else 2e-6) * scale
        base, off = ctypes.c_void_p(), ctypes.c_int64()
        for h in hs:
            ctx.check(ctx.lib.pq_tensor_device_ptr(ctx.ptr, h, ctypes.byref(base), ctypes.byref(off), None))
        for h, w in zip(hs, want):
            assert np.array_equal(ctx.download(h), w)
    finally:
        ctx.close()
