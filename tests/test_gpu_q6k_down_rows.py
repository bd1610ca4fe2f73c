"""Q6_K down rows of an odd number of super-blocks (every other row 2 bytes off a word boundary) on
the MFMA kernels, whole layers bit for bit against the oracle: one, three and five super-blocks, slot
tiles from one slot to full ones, both block shapes (under and from six slots per expert)."""
import numpy as np
import pytest

import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("F", [256, 768, 1280])
@pytest.mark.parametrize("T", [4, 9, 33, 64])
def test_q6k_down_odd_rows(F, T):
    from large_model_amd import qmsg
    E, X, K = 512, 16, 8
    print(f"[case] q6k odd rows F={F} T={T}", flush=True)
    L = orc.Layer(E, X, K, F, 30, down_type=orc.T_Q6_K)
    x = orc.make_input(E, T, 31)
    with qmsg.Context(E, X, K, F, max_tokens=T) as ctx:
        ctx.synth(0, 30, down_type=orc.T_Q6_K)
        outs = [ctx.moe(0, x)]
        ctx.set_path(qmsg.PATH_MFMA)               # also below the slots from which the default takes it
        outs.append(ctx.moe(0, x))
    want = L.moe(x)
    for out in outs:
        assert np.array_equal(out.view(np.uint32), want.view(np.uint32))
