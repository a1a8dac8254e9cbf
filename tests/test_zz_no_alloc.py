"""The allocation-free W4A8 entry point (rai_w4a8_matmul_noalloc_dev) against
rai_w4a8_matmul_dev, through the C ABI: bit-identical outputs on two calls in
a row on the same device buffers, the second with fewer tokens and a smaller
matrix (the shared scratch keeps the first call's contents), every kernel that
the route picks, also captured in a graph and replayed, and the size limit."""
import ctypes
import gc

import numpy as np
import pytest

from rai_amd.workload import gemv_operands

pytestmark = pytest.mark.gpu


def _run(rai, fn, nib, params, x, rows, cols, m, gs):
    L = rai.lib()
    dn, dp, dx = rai.DeviceArray.from_host(nib), rai.DeviceArray.from_host(params), rai.DeviceArray.from_host(x)
    do = rai.DeviceArray(4 * m * rows)
    rc = getattr(L, fn)(do.ptr, dn.ptr, dp.ptr, dx.ptr, rows, cols, m, gs, None)
    assert rc == 0, L.rai_last_error().decode()
    assert L.rai_device_synchronize() == 0
    return do.to_host(np.float32, m * rows).view(np.uint32)


@pytest.mark.parametrize("calls", [
    [(4096, 4096, 9, 32), (1024, 2048, 5, 32)],     # register-pipelined, then smaller
    [(2000, 4096, 16, 32), (300, 512, 1, 32)],      # then the one-token path
    [(512, 14336, 3, 32), (96, 1024, 2, 64)],       # long rows, then two tokens at group 64
    [(1000, 8192, 128, 128), (64, 256, 17, 32)],    # streamed, then a few short rows
    [(4096, 4096, 200, 32), (1024, 2048, 70, 32)],  # the matrix-core GEMM, then streamed
    [(16, 349472, 3, 32), (16, 349440, 3, 32)],     # streamed records past the scratch (VALU kernel), then inside it
])
def test_noalloc_matches_allocating_entry_point(rai, calls):
    for i, (rows, cols, m, gs) in enumerate(calls):
        nib, params, x = gemv_operands(rows, cols, m, gs, seed=rows + m + i)
        want = _run(rai, "rai_w4a8_matmul_dev", nib, params, x, rows, cols, m, gs)
        got = _run(rai, "rai_w4a8_matmul_noalloc_dev", nib, params, x, rows, cols, m, gs)
        assert np.array_equal(got, want), (i, rows, cols, m, gs)


@pytest.mark.parametrize("rows,cols,m,gs", [
    (300, 512, 1, 32), (300, 8192, 1, 64),  # one token: quantized in its GEMV, or before it
    (200, 1088, 2, 64),                     # tiled VALU kernel
    (1024, 2048, 9, 32),                    # register-pipelined
    (4096, 1152, 9, 128),                   # streamed
    (16384, 128, 70, 64),                   # GEMM
    (33, 100, 3, 40),                       # a ragged last group
])
def test_noalloc_in_a_graph(rai, rows, cols, m, gs):
    """Captured once and replayed on new inputs, with eager calls between the
    replays (they overwrite the shared scratch): each replay equals the eager
    call on its input."""
    L = rai.lib()
    nib, params, _ = gemv_operands(rows, cols, m, gs, seed=rows + m)
    xs = [gemv_operands(rows, cols, m, gs, seed=100 + i)[2] for i in range(3)]
    want = [_run(rai, "rai_w4a8_matmul_noalloc_dev", nib, params, x, rows, cols, m, gs) for x in xs]
    dn, dp = rai.DeviceArray.from_host(nib), rai.DeviceArray.from_host(params)
    dx, do = rai.DeviceArray.from_host(xs[0]), rai.DeviceArray(4 * m * rows)
    P = ctypes.c_void_p
    stream, graph, ex = P(), P(), P()

    def hip(name, *args):
        rc = getattr(L, name)(*args)  # the HIP runtime that the library is linked with
        assert rc == 0, (name, rc)

    hip("hipStreamCreate", ctypes.byref(stream))
    # No garbage collection in between: a device array that it frees (hipFree from
    # the capturing thread) would invalidate the capture.
    gc.collect()
    gc.disable()
    try:
        hip("hipStreamBeginCapture", stream, 1)  # thread-local
        rc = L.rai_w4a8_matmul_noalloc_dev(do.ptr, dn.ptr, dp.ptr, dx.ptr, rows, cols, m, gs, stream)
        hip("hipStreamEndCapture", stream, ctypes.byref(graph))
    finally:
        gc.enable()
    assert rc == 0, L.rai_last_error().decode()
    hip("hipGraphInstantiate", ctypes.byref(ex), graph, None, None, ctypes.c_size_t(0))
    for x, w in list(zip(xs, want)) + [(xs[0], want[0])]:
        x = np.ascontiguousarray(x, np.float32)
        assert L.rai_memcpy_h2d(dx.ptr, x.ctypes.data_as(P), x.nbytes) == 0
        hip("hipGraphLaunch", ex, stream)
        hip("hipStreamSynchronize", stream)
        assert np.array_equal(do.to_host(np.float32, m * rows).view(np.uint32), w)
        _run(rai, "rai_w4a8_matmul_noalloc_dev", nib, params, xs[1] * 3, rows, cols, m, gs)
    hip("hipGraphExecDestroy", ex)
    hip("hipGraphDestroy", graph)
    hip("hipStreamDestroy", stream)


def test_noalloc_rejects_sizes_past_the_scratch(rai):
    L = rai.lib()
    rows, cols, gs = 64, 4096, 32
    nib, params, x = gemv_operands(rows, cols, 1, gs, seed=1)
    dn, dp = rai.DeviceArray.from_host(nib), rai.DeviceArray.from_host(params)
    m = (1 << 20) // cols + 1
    dx = rai.DeviceArray(4 * m * cols)
    do = rai.DeviceArray(4 * m * rows)
    rc = L.rai_w4a8_matmul_noalloc_dev(do.ptr, dn.ptr, dp.ptr, dx.ptr, rows, cols, m, gs, None)
    assert rc == -2  # RAI_E_SHAPE
    assert "scratch" in L.rai_last_error().decode()
