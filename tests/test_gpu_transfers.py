# -*- coding: utf-8 -*-
"""Host transfers and device blocks of the C ABI: null host pointers are
refused, transfers arrive whole where the staging wraps, freed blocks are used
again, bounded, and given back."""

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


def _held(ctx):
    """(bytes of the live buffers, device bytes behind them, the pool and the
    packing scratch, bytes of the staging)."""
    outs = [ctypes.c_int64() for _ in range(11)]
    assert ctx._lib.rvc_mem_stats(ctx.handle, *[ctypes.byref(o) for o in outs]) == 0
    return outs[5].value, outs[8].value, outs[6].value


def test_staging_wraps(ctx):
    """Uploads that are not waited for fill the 4 MiB staging several times
    over; every one of them arrives, in pieces of ragged sizes."""
    rng = np.random.default_rng(0)
    sizes = [1, 3, 63, 64, 65, 1 << 18, (1 << 18) - 1, (1 << 18) + 1, 100001, 77] * 3
    arrs = [rng.standard_normal(n, dtype=np.float32) for n in sizes]
    ids = [ctx.upload(a) for a in arrs]
    assert _held(ctx)[2] == 4 << 20
    for a, i in zip(arrs, ids):
        np.testing.assert_array_equal(ctx.download(i, a.shape), a)
    odd = rng.integers(0, 256, 1237, dtype=np.uint8)  # a tail below 16 bytes
    b = ctx.upload(odd)
    np.testing.assert_array_equal(ctx.download(b, odd.shape, np.uint8), odd)
    for i in ids + [b]:
        ctx.free(i)


def test_freed_blocks_are_used_again(ctx):
    for n in (1, 1000, 1 << 16, 3 << 20):
        a = ctx.alloc(n)
        ctx.free(a)
        held = _held(ctx)[1]
        b = ctx.alloc(n)
        assert _held(ctx)[1] == held
        ctx.free(b)


def test_freed_blocks_are_bounded(ctx):
    """At most 128 MiB stay, the oldest go first, and none above 32 MiB."""
    ids = [ctx.alloc(5 << 20) for _ in range(10)]  # 20 MiB each
    for i in ids:
        ctx.free(i)
    live, held, _ = _held(ctx)
    assert live == 0 and 100 << 20 < held <= 128 << 20
    new = ctx.alloc(7 << 20)  # 28 MiB
    ctx.free(new)             # pushes out older blocks, and stays itself
    held = _held(ctx)[1]
    assert held <= 128 << 20
    new = ctx.alloc(7 << 20)
    assert _held(ctx)[1] == held
    ctx.free(new)
    big = ctx.alloc(9 << 20)  # 36 MiB
    assert _held(ctx)[1] == held + (36 << 20)
    ctx.free(big)
    assert _held(ctx)[1] == held


def test_failed_allocation_gives_the_pool_back(ctx):
    ctx.free(ctx.alloc(1 << 20))
    assert _held(ctx)[1] > 0
    out = ctypes.c_int64()
    assert ctx._lib.rvc_mem_alloc(ctx.handle, 1 << 50, ctypes.byref(out)) == -1
    assert _held(ctx)[1] == 0
    x = np.arange(300, dtype=np.float32)
    b = ctx.upload(x)  # and the engine goes on
    np.testing.assert_array_equal(ctx.download(b, x.shape), x)
    ctx.free(b)
