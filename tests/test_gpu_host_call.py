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
