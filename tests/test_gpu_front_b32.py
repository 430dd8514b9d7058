"""The operand rows of the 32-value types and F16 written by the router's
launch, against the pass of its own that a caller-routed call takes: the same
ids and weights through mi_moe_expert_ffn give the same bits, for both products'
forms (integer dots and GEMM), widths the router's launch takes (multiples of
64) and does not, token counts around its 16-token slabs and one and two of its
column groups, with the router on the same rows and on rows of its own.
"""
import numpy as np
import pytest

import mimoe as M
from test_gpu_shared_gb import _quant

pytestmark = pytest.mark.gpu

TYPES = {"q8_0": M.TYPE_Q8_0, "q5_0": M.TYPE_Q5_0, "q4_0": M.TYPE_Q4_0, "f16": M.TYPE_F16}


@pytest.mark.parametrize("D,T", [(64, 1), (64, 17), (96, 5), (320, 15), (320, 16), (320, 33), (2112, 3), (2112, 130), (2048, 700)])
@pytest.mark.parametrize("t", list(TYPES.values()), ids=list(TYPES))
def test_rows_of_the_router_launch(t, D, T):
    rng = np.random.default_rng(D + T)
    E, K, I = 20, 3, 64
    keep = []

    def tab(*shape):
        keep.append(M.to_device(np.ascontiguousarray(_quant(t, (rng.standard_normal(shape) * 0.08).astype(np.float32)))))
        return M.tensor(keep[-1], t, list(shape[::-1]))

    rw = M.to_device((rng.standard_normal((E, D)) * 0.1).astype(np.float32))
    L = M.make_layer(D, E, K, I, rw, None, tab(E, I, D), tab(E, I, D), tab(E, D, I), False, M.ACT_SILU)
    x, xr = (M.to_device(rng.standard_normal((T, D)).astype(np.float32)) for _ in range(2))
    out, sel, w = M.DeviceBuffer(4 * T * D), M.DeviceBuffer(4 * T * K), M.DeviceBuffer(4 * T * K)
    ctx = M.Context(0)
    ctx.reserve(T, D, I, E, K)
    r = M.Routing()
    r.sel, r.weights = sel.addr, w.addr
    for thr in (1, 1 << 30):
        ctx.set_gemm_threshold(thr)
        for own in (False, True):
            if own:
                M.check("forward", ctx.forward_router_input(L, x, xr, T, None, out, r))
            else:
                M.check("forward", ctx.forward(L, x, T, None, out, r))
            got = out.download(np.float32, (T, D))
            M.check("expert_ffn", ctx.expert_ffn(L, x, T, None, sel, sel, w, out))
            assert np.array_equal(got, out.download(np.float32, (T, D))), (thr, own)
    assert ctx.take_errors() == (0, 0)
    ctx.close()
