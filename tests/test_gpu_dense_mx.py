"""Dense products on the MFMA kernels at the edges of their tiles: row counts that end inside a
64- or 128-row block, token counts on both sides of every block shape's range, one and two staged
chunks, and input blocks outside the scaled range, bit for bit against the oracle's qms_matmul."""
import numpy as np
import pytest

import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def q():
    from large_model_amd import qmsg
    return qmsg


def bits(a):
    return np.ascontiguousarray(a).view(np.uint32)


def check(q, specs, cols, x, seed):
    ws = [orc.synth_mat(t, r, cols, seed + i) for i, (t, r) in enumerate(specs)]
    with q.Context(256, 16, 4, 128, max_tokens=1) as ctx:
        ids = [ctx.mat_upload(t, w, r, cols) for (t, r), w in zip(specs, ws)]
        ys = ctx.matmul_n(ids, x)
    for (t, r), w, y in zip(specs, ws, ys):
        assert np.array_equal(bits(y), bits(orc.matmul_q8(t, w, r, cols, x))), (t, r)


@pytest.mark.parametrize("T", [5, 8, 9, 12, 16, 17, 32, 33, 64, 65, 95, 96, 130])
@pytest.mark.parametrize("cols", [256, 512])
def test_dense_mx_edges(q, T, cols):
    """From 9 tokens on the calls' Q4_0 and Q6_K matrices take the MFMA kernels; the Q4_1 pair,
    one matrix under 128 rows, keeps the row kernels."""
    print(f"[case] dense mx C={cols} T={T}", flush=True)
    specs = [(orc.T_Q4_0, 128), (orc.T_Q4_0, 201), (orc.T_Q4_1, 191), (orc.T_Q4_1, 64)]
    if cols == 512:
        specs += [(orc.T_Q6_K, 129), (orc.T_Q6_K, 320)]
    check(q, specs, cols, orc.make_input(cols, T, 70), 71)


@pytest.mark.parametrize("type_,rows,cols,T", [(orc.T_Q4_0, 1024, 256, 1601), (orc.T_Q6_K, 1090, 512, 2050),
                                               (orc.T_Q4_0, 4160, 4096, 6), (orc.T_Q6_K, 8192, 2048, 5),
                                               (orc.T_Q6_K, 10240, 2048, 5), (orc.T_Q4_0, 256, 65536, 6),
                                               (orc.T_Q6_K, 704, 24576, 7)])
def test_dense_mx_large_grids(q, type_, rows, cols, T):
    """The block shapes of large grids, and few tokens on large matrices."""
    print(f"[case] dense mx large type {type_} {rows}x{cols} T={T}", flush=True)
    check(q, [(type_, rows)], cols, orc.make_input(cols, T, 80), 81)


@pytest.mark.parametrize("T", [9, 40, 70])
@pytest.mark.parametrize("type_", [orc.T_Q4_0, orc.T_Q4_1, orc.T_Q6_K])
def test_dense_mx_scaled_range(q, T, type_):
    """Input blocks whose scale is subnormal or tiny take the unscaled loop; the call after it,
    in range on the same context, the scaled one."""
    print(f"[case] dense mx range type {type_} T={T}", flush=True)
    cols, rows = 512, 130
    w = orc.synth_mat(type_, rows, cols, 90)
    x = orc.make_input(cols, T, 91)
    small = x.copy()
    small[::2] *= np.float32(1e-36)
    small[1] = 0.0
    with q.Context(256, 16, 4, 128, max_tokens=1) as ctx:
        i = ctx.mat_upload(type_, w, rows, cols)
        for v in (small, x):
            y = ctx.matmul_n([i], v)[0]
            assert np.array_equal(bits(y), bits(orc.matmul_q8(type_, w, rows, cols, v)))
