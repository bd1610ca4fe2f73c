"""The fp32-chain rows on the fp32 matrix cores (qmsg_chain.hip) at the edges of their tiles: row
counts around 16 and 64, input rows around 16 and 32, widths of odd block counts and of partly
filled staging chunks, every row type, bit for bit against the oracle's matmul_exact and moe."""
import numpy as np
import pytest

import expert_types as et
import oracle as orc

pytestmark = pytest.mark.gpu
TYPES = [orc.T_F32, orc.T_F16, orc.T_Q4_0, orc.T_Q4_1, orc.T_Q8_0, orc.T_Q6_K]


@pytest.fixture(scope="module")
def q():
    from large_model_amd import qmsg
    return qmsg


def bits(a):
    return np.ascontiguousarray(a).view(np.uint32)


@pytest.mark.parametrize("cols", [32, 96, 256, 800, 1056, 2048, 2304])
@pytest.mark.parametrize("T", [1, 2, 15, 16, 17, 32, 33])
def test_chain_dense_edges(q, cols, T):
    print(f"[case] chain dense C={cols} T={T}", flush=True)
    specs = [(t, r) for t in TYPES if t != orc.T_Q6_K or cols % 256 == 0 for r in (1, 63, 66)]
    ws = [et.expert_bytes(t, r, cols, 1, 40 + i) for i, (t, r) in enumerate(specs)]
    x = orc.make_input(cols, T, 41)
    x[0, :4] = [1e-42, -0.0, 3e37, -1e-39]            # subnormals, a negative zero, near overflow
    with q.Context(256, 16, 4, 128, max_tokens=1) as ctx:
        ctx.set_path(q.PATH_FP32)
        ids = [ctx.mat_upload(t, w, r, cols) for (t, r), w in zip(specs, ws)]
        ys = ctx.matmul_n(ids, x)
    ref = orc.matmul_n([(t, w, r, cols) for (t, r), w in zip(specs, ws)], x, exact=True)
    for (t, r), y, want in zip(specs, ys, ref):
        assert np.array_equal(bits(y), bits(want)), (t, r)


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_chain_non_finite(q, bad):
    """A non-finite input or scale reaches exactly the results that hold it."""
    print(f"[case] chain non-finite {bad}", flush=True)
    cols, T, rows = 288, 18, 70
    w = et.expert_bytes(orc.T_Q8_0, rows, cols, 1, 50).copy()
    w.reshape(rows, cols // 32, 34)[5, 3, :2] = np.array([bad], np.float16).view(np.uint8)
    x = orc.make_input(cols, T, 51)
    x[17, 100] = bad
    with q.Context(256, 16, 4, 128, max_tokens=1) as ctx:
        y = ctx.matmul_n([ctx.mat_upload(orc.T_Q8_0, w, rows, cols)], x)[0]
    want = orc.matmul_n([(orc.T_Q8_0, w, rows, cols)], x)[0]
    fine = ~np.isnan(want)
    assert np.array_equal(np.isnan(y), np.isnan(want))
    assert np.array_equal(bits(y)[fine], bits(want)[fine])


@pytest.mark.parametrize("T", [3, 18])
@pytest.mark.parametrize("type_", [orc.T_F32, orc.T_F16, orc.T_Q8_0])
def test_chain_subnormal_results(q, type_, T):
    """Chains whose products and sums are subnormal, pass through zero, or move between subnormal and
    normal step by step."""
    cols, rows = 288, 70
    print(f"[case] chain subnormal type {type_} T={T}", flush=True)
    rng = np.random.default_rng(52 + T)
    x = orc.make_input(cols, T, 53)
    if type_ == orc.T_F32:
        w = np.ldexp(rng.standard_normal((rows, cols)), rng.integers(-80, -50, (rows, cols))).astype(np.float32)
        w = np.ascontiguousarray(w).view(np.uint8).ravel()
        x *= np.ldexp(np.float32(1), rng.integers(-104, -75, x.shape)).astype(np.float32)
    else:
        w = et.expert_bytes(type_, rows, cols, 1, 54)                 # values or scales down to 2^-24
        if type_ == orc.T_F16:
            w = (w.view(np.float16) * np.float16(1e-3)).view(np.uint8)
        x *= np.ldexp(np.float32(1), rng.integers(-136, -113 if type_ == orc.T_F16 else -125, x.shape)).astype(np.float32)
    x[1] = -x[0]
    want = orc.matmul_n([(type_, w, rows, cols)], x, exact=True)[0]
    small = np.abs(want) < np.finfo(np.float32).tiny
    assert (small & (want != 0)).mean() > 0.3                         # most results are themselves subnormal
    with q.Context(256, 16, 4, 128, max_tokens=1) as ctx:
        ctx.set_path(q.PATH_FP32)
        y = ctx.matmul_n([ctx.mat_upload(type_, w, rows, cols)], x)[0]
    assert np.array_equal(bits(y), bits(want))


@pytest.mark.parametrize("T", [1, 5, 16, 17, 40, 64, 65, 70])
@pytest.mark.parametrize("types", [(orc.T_Q8_0,) * 3, (orc.T_F16,) * 3, (orc.T_Q8_0, orc.T_F16, orc.T_Q8_0)])
def test_chain_layer(q, T, types):
    """Few experts, so that slot tiles hold 16, 17, 32 and a tail of slots; 128 and 130 slots are sorted by
    one wave and by sixteen."""
    E, X, K, F = 288, 4, 2, 96
    print(f"[case] chain layer {types} T={T}", flush=True)
    L = et.typed_layer(E, X, K, F, types, 60)
    x = orc.make_input(E, T, 61)
    with q.Context(E, X, K, F, max_tokens=T) as ctx:
        ctx.upload(0, L.router, (types[0], L.gate), (types[1], L.up), (types[2], L.down))
        out = ctx.moe(0, x)
    assert np.array_equal(bits(out), bits(L.moe(x)))


def test_chain_layer_many_tiles():
    """More slot tiles than a grid's y takes (65535): one large call against the same tokens in parts."""
    E, X, K, F, T = 32, 64, 64, 32, 33000
    print(f"[case] chain layer {T} tokens x {K} experts", flush=True)
    from large_model_amd import qmsg
    L = et.typed_layer(E, X, K, F, (orc.T_Q8_0,) * 3, 62)
    x = orc.make_input(E, T, 63)
    with qmsg.Context(E, X, K, F, max_tokens=T) as ctx:
        ctx.upload(0, L.router, *((orc.T_Q8_0, w) for w in (L.gate, L.up, L.down)))
        out = ctx.moe(0, x)
        parts = np.concatenate([ctx.moe(0, x[i:i + 11000]) for i in range(0, T, 11000)])
    assert np.array_equal(bits(out), bits(parts))
    assert np.array_equal(bits(out[-8:]), bits(L.moe(x[-8:])))


@pytest.mark.parametrize("T", [11, 12])
def test_chain_layer_staging(q, T):
    """Gate/up inputs of 1024 floats on both sides of the LDS that two blocks share."""
    E, X, K, F = 1024, 4, 2, 96
    print(f"[case] chain layer staging T={T}", flush=True)
    types = (orc.T_Q8_0,) * 3
    L = et.typed_layer(E, X, K, F, types, 66)
    x = orc.make_input(E, T, 67)
    with q.Context(E, X, K, F, max_tokens=T) as ctx:
        ctx.upload(0, L.router, *zip(types, (L.gate, L.up, L.down)))
        out = ctx.moe(0, x)
    assert np.array_equal(bits(out), bits(L.moe(x)))
