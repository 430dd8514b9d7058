"""The shared expert inside the routed experts' grouped GEMM launches, against
the same two parts run by themselves: the routed sum without a shared expert,
and the shared expert as a one-expert layer on mi_moe_expert_ffn (which runs
the same arithmetic in launches of its own).  Both are fp32 values the forward
adds once, so the sum is bit for bit; with a scalar gate row the weight is an
fp32 sigmoid, computed here in fp64: two ulp of the weight times the value.
Token counts around the 32- and 128-row tiles, each run on both; shared widths
with an odd number of blocks and more than a work-group's columns, tables the
launch cannot share (another type, another activation) beside those it can.
"""
import ctypes as C

import numpy as np
import pytest

import mimoe as M
import pyoracle as O

pytestmark = pytest.mark.gpu

D, E, K = 160, 6, 2


def _quant(t, w):
    w2 = w.reshape(-1, w.shape[-1])
    return w2.astype(np.float16).view(np.uint8) if t == M.TYPE_F16 else O.quantize(t, w2)


def _layer(rng, t, td, I, act, sh_I, sh_t, sh_td, sh_act, gate_row, keep):
    def tab(tt, *shape):
        buf = M.to_device(np.ascontiguousarray(_quant(tt, (rng.standard_normal(shape) * 0.08).astype(np.float32))))
        keep.append(buf)
        return M.tensor(buf, tt, list(shape[::-1]))

    rw = M.to_device((rng.standard_normal((E, D)) * 0.1).astype(np.float32))
    keep.append(rw)
    gated, sh_gated = act != M.ACT_RELU_SQR, sh_act != M.ACT_RELU_SQR
    L = M.make_layer(D, E, K, I, rw, None, tab(t, E, I, D), tab(t, E, I, D) if gated else None, tab(td, E, D, I), False, act)
    sg, su, sd = tab(sh_t, 1, sh_I, D), tab(sh_t, 1, sh_I, D) if sh_gated else None, tab(sh_td, 1, D, sh_I)
    one = M.make_layer(D, 1, 1, sh_I, None, None, sg, su, sd, False, sh_act)
    with_sh = M.Layer.from_buffer_copy(L)
    with_sh.sh_n_ff, with_sh.sh_act, with_sh.sh_gate, with_sh.sh_down = sh_I, sh_act, sg, sd
    if su is not None:
        with_sh.sh_up = su
    if gate_row is not None:
        keep.append(M.to_device(gate_row))
        with_sh.sh_gate_inp = C.c_void_p(keep[-1].addr)
    return L, one, with_sh


CASES = [  # routed gate / down types, act, shared gate / down types, act
    (M.TYPE_Q8_0, M.TYPE_Q8_0, M.ACT_SILU, M.TYPE_Q8_0, M.TYPE_Q8_0, M.ACT_SILU),
    (M.TYPE_Q5_0, M.TYPE_Q5_0, M.ACT_RELU_SQR, M.TYPE_Q5_0, M.TYPE_Q5_0, M.ACT_RELU_SQR),
    (M.TYPE_Q4_0, M.TYPE_F16, M.ACT_GELU_TANH, M.TYPE_Q4_0, M.TYPE_F16, M.ACT_GELU_TANH),
    (M.TYPE_F16, M.TYPE_F16, M.ACT_SILU, M.TYPE_F16, M.TYPE_F16, M.ACT_SILU),
    (M.TYPE_Q8_0, M.TYPE_Q8_0, M.ACT_SILU, M.TYPE_Q8_0, M.TYPE_F16, M.ACT_SILU),
    (M.TYPE_Q8_0, M.TYPE_Q8_0, M.ACT_SILU, M.TYPE_Q8_0, M.TYPE_Q8_0, M.ACT_GELU_ERF),
]


@pytest.mark.parametrize("gated_row", [False, True], ids=["", "gate_row"])
@pytest.mark.parametrize("case", CASES, ids=["q8_0", "q5_0_relu2", "q4_0_f16", "f16", "other_type", "other_act"])
@pytest.mark.parametrize("T,sh_I", [(2, 32), (31, 96), (33, 288), (128, 416), (129, 96), (300, 1056)])
def test_shared_in_the_routed_launches(T, sh_I, case, gated_row):
    t, td, act, sh_t, sh_td, sh_act = case
    rng = np.random.default_rng(T + sh_I)
    keep, I = [], 96
    gate_row = (rng.standard_normal(D) * 0.1).astype(np.float32) if gated_row else None
    L, one, with_sh = _layer(rng, t, td, I, act, sh_I, sh_t, sh_td, sh_act, gate_row, keep)
    x = rng.standard_normal((T, D)).astype(np.float32)
    w = np.ones((T, 1), np.float32)
    ulp = 0
    if gated_row:
        # a one-expert router row: its fp32 logit to within an ulp of fp64
        w = (1.0 / (1.0 + np.exp(-(x.astype(np.float64) @ gate_row.astype(np.float64)))))[:, None].astype(np.float32)
        ulp = 2
    ctx = M.Context(0)
    ctx.reserve(T, D, max(I, sh_I), E, K)
    ctx.set_gemm_threshold(1)
    xd, out = M.to_device(x), M.DeviceBuffer(4 * T * D)

    def get():
        return out.download(np.float32, (T, D))

    M.check("forward", ctx.forward(L, xd, T, None, out))
    routed = get()
    ids, wd = M.to_device(np.zeros((T, 1), np.int32)), M.to_device(w)
    M.check("expert_ffn", ctx.expert_ffn(one, xd, T, None, ids, ids, wd, out))
    shared = get()
    M.check("forward", ctx.forward(with_sh, xd, T, None, out))
    got = get()
    for kind in (1, 2):   # 128- and 32-row tiles throughout
        ctx.set_gemm_tiles(kind)
        M.check("forward", ctx.forward(with_sh, xd, T, None, out))
        assert np.array_equal(get().view(np.uint32), got.view(np.uint32)), kind
    assert ctx.take_errors() == (0, 0)
    ctx.close()
    want = routed + shared
    # ulp steps of the weight on the shared value, then one rounding of the sum
    lim = 0.0 if not ulp else ulp * 2.0 ** -23 * np.abs(shared) + 2.0 ** -23 * np.abs(want)
    assert np.all(np.abs(got - want) <= lim), (np.abs(got - want).max(), np.abs(want).max())
