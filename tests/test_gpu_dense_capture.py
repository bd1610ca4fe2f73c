"""Dense calls captured into a HIP graph: replays after larger eager calls, which replace the
context's record buffer, keep the eager call's bits."""
import ctypes

import numpy as np
import pytest

import oracle as orc

pytestmark = pytest.mark.gpu


def hip_lib():
    hip, vp = ctypes.CDLL("libamdhip64.so"), ctypes.c_void_p
    hip.hipStreamBeginCapture.argtypes = [vp, ctypes.c_int]
    hip.hipStreamEndCapture.argtypes = [vp, ctypes.POINTER(vp)]
    hip.hipGraphInstantiate.argtypes = [ctypes.POINTER(vp), vp, vp, vp, ctypes.c_size_t]
    hip.hipGraphLaunch.argtypes = [vp, vp]
    hip.hipGraphExecDestroy.argtypes = [vp]
    hip.hipGraphDestroy.argtypes = [vp]
    return hip


@pytest.mark.parametrize("T", [5, 7, 8, 16])
def test_capture_survives_growth(T):
    from large_model_amd import qmsg
    hip, vp = hip_lib(), ctypes.c_void_p
    rows, cols, big = 4160, 4096, 64                  # rows * cols >= 2^24: eager calls take the MFMA kernels
    print(f"[case] captured dense call T={T}", flush=True)
    x = orc.make_input(cols, big, 20)
    w = orc.synth_mat(orc.T_Q4_0, rows, cols, 21)
    want = orc.matmul_q8(orc.T_Q4_0, w, rows, cols, x)
    with qmsg.Context(256, 16, 4, 128, max_tokens=1) as ctx:
        i = ctx.mat_upload(orc.T_Q4_0, w, rows, cols)
        st = vp(qmsg.lib.qmsg_stream(ctx._h))
        d_x, d_y = ctx.device_alloc(4 * x.nbytes), ctx.device_alloc(T * rows * 4)
        d_yb = ctx.device_alloc(4 * want.nbytes)
        ctx.h2d(d_x, np.tile(x, (4, 1)))
        ctx.matmul_n_device([i], d_x, T + 8, [d_yb])  # leaves a buffer that holds T rows
        ctx.sync()
        graph, exe = vp(), vp()
        assert hip.hipStreamBeginCapture(st, 2) == 0  # relaxed capture mode
        ctx.matmul_n_device([i], d_x, T, [d_y])
        assert hip.hipStreamEndCapture(st, ctypes.byref(graph)) == 0
        assert hip.hipGraphInstantiate(ctypes.byref(exe), graph, None, None, 0) == 0
        try:
            for n in (32, big, 2 * big, 4 * big):     # each larger call replaces the buffer
                ctx.matmul_n_device([i], d_x, n, [d_yb])
                ctx.h2d(d_y, np.zeros((T, rows), np.float32))
                assert hip.hipGraphLaunch(exe, st) == 0
                ctx.sync()
                assert np.array_equal(ctx.d2h(d_y, (T, rows)).view(np.uint32), want[:T].view(np.uint32)), n
                m = min(n, big)
                assert np.array_equal(ctx.d2h(d_yb, (m, rows)).view(np.uint32), want[:m].view(np.uint32)), n
        finally:
            hip.hipGraphExecDestroy(exe)
            hip.hipGraphDestroy(graph)
