"""One token with the caller's expert ids and weights (mi_moe_expert_ffn) on
the fused single-token kernel, through the C ABI, against the CPU oracle and
the kernel chain: separate gate/up and down ids, repeated ids, ids outside
[0, E) (their slots left out, counted), 1 to 8 slots, Q4_K and Q6_K down,
fused and separate tables, the forced rescue path bit for bit, out over res,
and out over x (which runs the chain).

Bar: 1e-4 against the oracle (both sides take exact integer dots; an fp32 GLU
value that differs in its last bit may move one Q8_K code of a block of 256,
1 / 127 of its maximum in one of 256 x K values).
"""
import numpy as np
import pytest

import mimoe as M
import pyoracle as O
from _util import rel_l2

pytestmark = pytest.mark.gpu


class Layer:
    def __init__(self, D, I, E, K, fused, td, seed):
        rng = np.random.default_rng(seed)
        f = lambda *s: (rng.standard_normal(s) * 0.03).astype(np.float32)  # noqa: E731
        q = lambda t, a: O.quantize(t, a.reshape(-1, a.shape[-1])).reshape(a.shape[:-1] + (-1,))  # noqa: E731
        gate, up, down = q(M.TYPE_Q4_K, f(E, 2 * I if fused else I, D)), q(M.TYPE_Q4_K, f(E, I, D)), q(td, f(E, D, I))
        act = M.ACT_GELU_ERF_GP1 if fused else M.ACT_SILU
        self.dims = (D, I, E, K)
        self.o = dict(D=D, E=E, K=K, I=I, router_w=np.zeros((E, D), np.float32), router_b=None, gate=gate,
                      up=None if fused else up, down=down, gate_type=M.TYPE_Q4_K, down_type=td, fused=fused, act=act,
                      gating=M.GATING_SOFTMAX_TOPK)
        self.dev = [M.to_device(a) for a in (gate, up, down)]
        self.L = M.make_layer(D, E, K, I, None, None, M.tensor(self.dev[0], M.TYPE_Q4_K, [D, gate.shape[1], E]),
                              None if fused else M.tensor(self.dev[1], M.TYPE_Q4_K, [D, I, E]),
                              M.tensor(self.dev[2], td, [I, D, E]), fused, act)
        self.x = rng.standard_normal((1, D)).astype(np.float32)
        self.res = rng.standard_normal((1, D)).astype(np.float32)
        self.w = (rng.random((1, K)) + 0.2).astype(np.float32)
        self.ctx = M.Context(0)
        self.ctx.reserve(1, D, I, E, K)

    def run(self, gu, dn=None, res=True, mode=M.DECODE_FUSED, rescue=64, alias=None):
        D = self.dims[0]
        c = self.ctx
        c.set_fused_decode(mode)
        c.set_decode_rescue(rescue)
        xd, rd, wd = M.to_device(self.x), M.to_device(self.res), M.to_device(self.w)
        gd = M.to_device(np.asarray(gu, np.int32))
        dd = gd if dn is None else M.to_device(np.asarray(dn, np.int32))
        out = rd if alias == "res" else xd if alias == "x" else M.DeviceBuffer(4 * D)
        M.check("expert_ffn", c.expert_ffn(self.L, xd, 1, rd if res else None, gd, dd, wd, out))
        return out.download(np.float32, (1, D))

    def ref(self, gu, dn=None, res=True):
        return O.moe_forward(self.o, self.x, self.res if res else None, sel_in=np.asarray(gu, np.int32).reshape(1, -1), w_in=self.w,
                             down_sel_in=None if dn is None else np.asarray(dn, np.int32).reshape(1, -1))[0]


@pytest.mark.parametrize("D,I,E,K,fused,td", [
    (2048, 768, 128, 8, False, M.TYPE_Q4_K), (2048, 1024, 64, 8, True, M.TYPE_Q6_K), (256, 256, 4, 1, True, M.TYPE_Q4_K),
    (512, 256, 256, 3, False, M.TYPE_Q6_K),
    # (2 K < E throughout: the chain takes its exact GEMV, not the fp16 GEMM)
    (1024, 2048, 8, 2, True, M.TYPE_Q4_K)],
    ids=["qwen3omni", "moondream3", "one_slot", "e256", "long_down"])
def test_caller_ids(D, I, E, K, fused, td):
    l = Layer(D, I, E, K, fused, td, seed=D + I)
    rng = np.random.default_rng(1)
    gu, dn = rng.permutation(E)[:K], rng.integers(0, E, K)
    for d in (None, dn):
        ref = l.ref(gu, d)
        got = l.run(gu, d)
        e = rel_l2(got - l.res, ref - l.res)
        print(f"D={D} I={I} K={K} down ids {'same' if d is None else 'own'}: {e:.2e}", flush=True)
        assert e <= 1e-4
        assert rel_l2(l.run(gu, d, mode=M.DECODE_CHAIN) - l.res, got - l.res) <= 1e-4
        for polls in (0, 1):
            assert np.array_equal(l.run(gu, d, rescue=polls).view(np.uint32), got.view(np.uint32))
        assert np.array_equal(l.run(gu, d, alias="res").view(np.uint32), got.view(np.uint32))
        assert rel_l2(l.run(gu, d, alias="x") - l.res, ref - l.res) <= 1e-4
    assert rel_l2(l.run(gu, res=False), l.ref(gu, res=False)) <= 1e-4
    assert l.ctx.take_errors() == (0, 0)
    l.ctx.close()


def test_repeated_and_bad_ids():
    l = Layer(2048, 768, 16, 8, False, M.TYPE_Q4_K, seed=9)
    gu = np.array([3, 3, 5, 16, 0, -1, 3, 15])
    live = np.array([0, 1, 2, 4, 6, 7])
    w = l.w.copy()
    good = gu.copy()
    good[[3, 5]] = 0
    l.w[0, [3, 5]] = 0.0
    ref = l.ref(good)
    l.w[:] = w
    l.w[0, 3] = np.inf            # a dead slot's weight does not reach the sum
    got = l.run(gu)
    assert l.ctx.take_errors()[0] == 2 and len(live) == 6
    assert rel_l2(got - l.res, ref - l.res) <= 1e-4
    # separate down ids: a slot with either id outside is dead, every bad id is counted
    dn = np.array([1, 2, 16, 4, 5, 99, 7, 8])
    l.w[:] = w
    ok = (gu >= 0) & (gu < 16) & (dn < 16)
    l.w[0, ~ok] = 0.0
    ref = l.ref(np.where(ok, gu, 0), np.where(ok, dn, 0))
    l.w[:] = w
    got = l.run(gu, dn)
    assert l.ctx.take_errors()[0] == 4
    assert rel_l2(got - l.res, ref - l.res) <= 1e-4
    l.ctx.close()


def test_two_tokens():
    # a launch per token: bit for bit the two single calls; out over res too
    l = Layer(2048, 768, 64, 8, False, M.TYPE_Q4_K, seed=21)
    D, I, E, K = l.dims
    rng = np.random.default_rng(2)
    x, res = rng.standard_normal((2, D)).astype(np.float32), rng.standard_normal((2, D)).astype(np.float32)
    ids = np.stack([rng.permutation(E)[:K] for _ in range(2)]).astype(np.int32)
    w = (rng.random((2, K)) + 0.2).astype(np.float32)
    l.ctx.reserve(2, D, I, E, K)
    one = np.zeros((2, D), np.float32)
    for t in range(2):
        l.x, l.res, l.w = x[t:t + 1], res[t:t + 1], w[t:t + 1]
        one[t] = l.run(ids[t])[0]
    for alias in (False, True):
        xd, rd, idd, wd = M.to_device(x), M.to_device(res), M.to_device(ids), M.to_device(w)
        out = rd if alias else M.DeviceBuffer(8 * D)
        M.check("expert_ffn", l.ctx.expert_ffn(l.L, xd, 2, rd, idd, idd, wd, out))
        assert np.array_equal(out.download(np.uint32, (2, D)), one.view(np.uint32))
    l.ctx.close()
