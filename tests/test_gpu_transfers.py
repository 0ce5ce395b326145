# -*- coding: utf-8 -*-
"""Host transfers of the C ABI: null host pointers are refused, small and large
transfers arrive whole whatever the order of calls."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

F32P = ctypes.POINTER(ctypes.c_float)


@pytest.fixture()
def ctx():
    from rvc_hip import _hip, hip_ops

    assert _hip.has_so, _hip.so_load_error
    c = hip_ops.HipContext()
    yield c
    c.close()


@pytest.mark.parametrize("n", [1, 1 << 10, 1 << 20])
def test_null_host_pointers_are_refused(ctx, n):
    """Up to 1 MiB goes through the staging, above straight to the caller."""
    L, h, out = ctx._lib, ctx.handle, ctypes.c_int64(7)
    x = np.arange(n, dtype=np.float32)
    b = ctx.upload(x)
    assert L.rvc_mem_upload(h, None, n, ctypes.byref(out)) == -1 and out.value == 7
    assert L.rvc_mem_upload_bytes(h, None, 4 * n, ctypes.byref(out)) == -1 and out.value == 7
    assert L.rvc_mem_upload_to(h, None, n, b) == -1
    assert L.rvc_mem_download(h, b, None, n) == -1
    assert L.rvc_mem_download_bytes(h, b, None, 4 * n) == -1
    # nothing to move: a null pointer is as good as any
    assert L.rvc_mem_upload(h, None, 0, ctypes.byref(out)) == 0
    ctx.free(out.value)
    assert L.rvc_mem_upload_to(h, None, 0, b) == 0 and L.rvc_mem_download(h, b, None, 0) == 0
    np.testing.assert_array_equal(ctx.download(b, x.shape), x)
