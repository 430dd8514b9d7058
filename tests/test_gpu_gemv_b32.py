"""The grouped GEMV of the 32-value types and F16 tables: its own reading of
the router's ids (against the dispatch's lists, which a call that asks for the
counts takes), the tokens of an expert by ones, twos and fours, widths of less
than a pass over the lanes and past one LDS slice, and the shared expert in the
same launches (against the same two parts run by themselves).  All of these
are the same sums in the same order: bit for bit.  Against the oracle (the
activations' Q8_0 codes exact, fp32 sums of K / 32 block terms in eight chains
against its one): 1e-4.
"""
import numpy as np
import pytest

import mimoe as M
import pyoracle as O
from _util import rel_l2
from test_gpu_shared_gb import _quant

pytestmark = pytest.mark.gpu

NAMES = {M.TYPE_Q8_0: "q8_0", M.TYPE_Q5_0: "q5_0", M.TYPE_Q4_0: "q4_0", M.TYPE_F16: "f16"}


def _run(t, td, D, I, E, K, T, act, sh_I=0, seed=0):
    rng = np.random.default_rng(seed)
    keep = []
    gated = act != M.ACT_RELU_SQR

    def tab(tt, *shape):
        rows = np.ascontiguousarray(_quant(tt, (rng.standard_normal(shape) * 0.08).astype(np.float32)))
        keep.append(M.to_device(rows))
        return M.tensor(keep[-1], tt, list(shape[::-1])), rows

    gate, gate_r = tab(t, E, I, D)
    up, up_r = tab(t, E, I, D) if gated else (None, None)
    down, down_r = tab(td, E, D, I)
    rw = (rng.standard_normal((E, D)) * 0.1).astype(np.float32)
    keep.append(M.to_device(rw))
    L = M.make_layer(D, E, K, I, keep[-1], None, gate, up, down, False, act)
    x = rng.standard_normal((T, D)).astype(np.float32)
    ctx = M.Context(0)
    ctx.reserve(T, D, max(I, sh_I), E, K)
    ctx.set_gemm_threshold(1 << 30)
    xd, out, counts = M.to_device(x), M.DeviceBuffer(4 * T * D), M.DeviceBuffer(4 * E)
    got = {}
    for name in ("ids", "lists"):
        r = None
        if name == "lists":
            r = M.Routing()
            r.counts = counts.addr
        M.check("forward", ctx.forward(L, xd, T, None, out, r))
        got[name] = out.download(np.float32, (T, D))
    assert np.array_equal(got["ids"], got["lists"])
    assert counts.download(np.int32, (E,)).sum() == T * K
    o = dict(D=D, E=E, K=K, I=I, router_w=rw, router_b=None, gate=gate_r.ravel(), up=up_r.ravel() if gated else None,
             down=down_r.ravel(), gate_type=t, down_type=td, fused=False, act=act, gating=M.GATING_SOFTMAX_TOPK)
    ref, _ = O.moe_forward(o, x, None)
    e = rel_l2(got["ids"], ref)
    print(f"{NAMES[t]}/{NAMES[td]} D={D} I={I} E={E} K={K} T={T}: {e:.2e}", flush=True)
    if sh_I:
        sg, _ = tab(t, 1, sh_I, D)
        su = tab(t, 1, sh_I, D)[0] if gated else None
        sd, _ = tab(td, 1, D, sh_I)
        one = M.make_layer(D, 1, 1, sh_I, None, None, sg, su, sd, False, act)
        L.sh_n_ff, L.sh_act, L.sh_gate, L.sh_down = sh_I, act, sg, sd
        if gated:
            L.sh_up = su
        ids, wd = M.to_device(np.zeros((T, 1), np.int32)), M.to_device(np.ones((T, 1), np.float32))
        M.check("expert_ffn", ctx.expert_ffn(one, xd, T, None, ids, ids, wd, out))
        want = got["ids"] + out.download(np.float32, (T, D))
        M.check("forward", ctx.forward(L, xd, T, None, out))
        assert np.array_equal(out.download(np.float32, (T, D)), want)
    assert ctx.take_errors() == (0, 0)
    ctx.close()
    return e


@pytest.mark.parametrize("T", [1, 2, 3, 5, 8, 9, 33, 256, 300])
@pytest.mark.parametrize("t", list(NAMES), ids=NAMES.values())
def test_rows_from_the_ids(t, T):
    # 3 experts of which 2 are used: up to 200 rows each, at T = 300 past the ids a work-group reads
    assert _run(t, t, 160, 96, 3, 2, T, M.ACT_SILU, sh_I=96 if T < 40 else 0, seed=T) <= 1e-4


@pytest.mark.parametrize("D,I,sh_I", [(32, 32, 64), (256, 288, 32), (4160, 96, 160), (224, 4128, 0)])
@pytest.mark.parametrize("t,td", [(t, t) for t in NAMES] + [(M.TYPE_F16, M.TYPE_Q8_0), (M.TYPE_Q5_0, M.TYPE_F16)],
                         ids=[*NAMES.values(), "f16-q8_0", "q5_0-f16"])
def test_widths(t, td, D, I, sh_I):
    assert _run(t, td, D, I, 9, 3, 4, M.ACT_GELU_TANH, sh_I, seed=D) <= 3e-4   # (a code of a GLU value on an edge: 1 / 127)
    assert _run(t, td, D, I, 9, 3, 7, M.ACT_RELU_SQR, sh_I, seed=I) <= 3e-4
