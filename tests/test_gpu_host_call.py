"""The layer call on host buffers, on both sides of the size from which it takes pageable copies
instead of pinned rows, repeated on one context, and after a refused call: the device call's bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_host_call_sizes():
    from large_model_amd import qmsg
    E, X, K, F = 1024, 16, 4, 128
    rng = np.random.default_rng(5)
    print("[case] host call sizes", flush=True)
    with qmsg.Context(E, X, K, F, n_layer=2, max_tokens=80) as ctx:
        for l in range(2):
            ctx.synth(l, 40 + l)
        d_x, d_y = ctx.device_alloc(80 * E * 4), ctx.device_alloc(80 * E * 4)
        for T in (1, 64, 65, 2, 80, 3):                   # 64 rows of 1024 floats are 256 KiB
            for l in range(2):
                x = rng.standard_normal((T, E)).astype(np.float32)
                out = ctx.moe(l, x)
                ctx.h2d(d_x, x)
                ctx.moe_device(l, d_x, T, d_y)
                want = ctx.d2h(d_y, (T, E))
                assert np.array_equal(out.view(np.uint32), want.view(np.uint32)), (T, l)
                with pytest.raises(qmsg.QmsgError):
                    ctx.moe(2, x[:1])


def test_copy_launch_sizes():
    """The copy launch's grid follows the bytes: none, one unit, a block and one more, past its 4096 blocks."""
    from large_model_amd import qmsg
    print("[case] copy launch sizes", flush=True)
    n = 4096 * 256 * 16 + 4096
    x = np.random.default_rng(6).integers(0, 256, n, dtype=np.uint8)
    with qmsg.Context(256, 16, 4, 128) as ctx:
        d_x, d_y = ctx.device_alloc(n), ctx.device_alloc(n)
        ctx.h2d(d_x, x)
        for b in (0, 16, 4096, 4112, n):
            ctx.h2d(d_y, np.zeros(n, np.uint8))
            ctx._check(qmsg.lib.qmsg_calibrate_copy(ctx._h, d_y, d_x, b))
            y = ctx.d2h(d_y, (n,), np.uint8)
            assert np.array_equal(y[:b], x[:b]) and not y[b:].any(), b
