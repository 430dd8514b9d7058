"""Q6_K gate/up tables on the 4-wave grouped GEMMs, through the C ABI against
the CPU oracle: both tile sizes bit for bit the same, rows whose blocks start
at every even byte (odd block counts: 210 bytes a block), fused and separate
tables, Q4_K and Q6_K down, tiles at 1, 31-33 and 191-193 rows; a tiled copy of
the down table (the bits of the call without it); the 32-row tiles that find
their rows from the router's ids, against the dispatch's lists (which a call
that asks for the counts takes); and the tables those GEMMs do not take (gate
and up rows at different strides), which run the 16-row GEMM and agree to the
fp32 order of the sums and the Q8_K steps it moves.

Bars: 1e-2 against the oracle (fp16 operands, and one step of a Q8_K code
where a GLU value lies on the edge of two); between the two GEMMs the same
products summed in another order: a GLU value moves by ~1e-7, which moves a
Q8_K code of a block of 256 by one step (1 / 127 of its maximum) for ~1e-4 of
the values: 2e-3.
"""
import numpy as np
import pytest

import mimoe as M
import pyoracle as O
from _util import rel_l2

pytestmark = pytest.mark.gpu


def _run(D, I, E, K, T, fused, td, up_pad=0, kinds=(1, 2), seed=0, ids=None):
    rng = np.random.default_rng(seed)
    f = lambda *s: (rng.standard_normal(s) * 0.03).astype(np.float32)  # noqa: E731
    q = lambda t, a: O.quantize(t, a.reshape(-1, a.shape[-1])).reshape(a.shape[:-1] + (-1,))  # noqa: E731
    gate = q(M.TYPE_Q6_K, f(E, 2 * I if fused else I, D))
    up = q(M.TYPE_Q6_K, f(E, I, D))
    down = q(td, f(E, D, I))
    x = rng.standard_normal((T, D)).astype(np.float32)
    if ids is None:
        ids = np.stack([rng.permutation(E)[:K] for _ in range(T)]).astype(np.int32)
    w = rng.random((T, K)).astype(np.float32) + 0.5
    rb = gate.shape[-1]
    upp = np.zeros((E, I, rb + up_pad), np.uint8)
    upp[:, :, :rb] = up
    dev = [M.to_device(a) for a in (gate, upp, down, x, ids, w)]
    L = M.make_layer(D, E, K, I, None, None, M.tensor(dev[0], M.TYPE_Q6_K, [D, gate.shape[1], E]),
                     None if fused else M.tensor(dev[1], M.TYPE_Q6_K, [D, I, E],
                                                 [210, rb + up_pad, (rb + up_pad) * I, (rb + up_pad) * I * E]),
                     M.tensor(dev[2], td, [I, D, E]), fused, M.ACT_GELU_ERF_GP1 if fused else M.ACT_SILU)
    ctx = M.Context(0)
    ctx.reserve(T, D, I, E, K)
    ctx.set_gemm_threshold(1)
    out = M.DeviceBuffer(4 * T * D)
    got = []
    for kind in kinds:
        ctx.set_gemm_tiles(kind)
        M.check("expert_ffn", ctx.expert_ffn(L, dev[3], T, None, dev[4], dev[4], dev[5], out))
        got.append(out.download(np.float32, (T, D)))
    assert ctx.take_all_errors() == (0, 0, 0)
    ctx.close()
    o = dict(D=D, E=E, K=K, I=I, router_w=np.zeros((E, D), np.float32), router_b=None, gate=gate, up=None if fused else up,
             down=down, gate_type=M.TYPE_Q6_K, down_type=td, fused=fused,
             act=M.ACT_GELU_ERF_GP1 if fused else M.ACT_SILU, gating=M.GATING_SOFTMAX_TOPK)
    ref, _ = O.moe_forward(o, x, None, sel_in=ids, w_in=w)
    e = rel_l2(got[0], ref)
    print(f"D={D} I={I} T={T} fused={fused} down {td} pad {up_pad}: {e:.2e}", flush=True)
    assert e <= 1e-2
    for g in got[1:]:
        assert np.array_equal(g.view(np.uint32), got[0].view(np.uint32))
    return got[0]


@pytest.mark.parametrize("td", [M.TYPE_Q6_K, M.TYPE_Q4_K], ids=["q6_k", "q4_k"])
@pytest.mark.parametrize("fused", [True, False], ids=["fused", "separate"])
@pytest.mark.parametrize("D,I,T", [(256, 256, 5), (768, 256, 70), (1280, 512, 33), (2048, 768, 200)])
def test_shapes(D, I, T, fused, td):
    _run(D, I, 5, 2, T, fused, td, seed=D + T)


@pytest.mark.parametrize("rows", [1, 31, 32, 33, 191, 192, 193, 400])
def test_tile_rows(rows):
    ids = np.array([0] * rows + [1], np.int32).reshape(-1, 1)
    _run(256, 256, 3, 1, rows + 1, True, M.TYPE_Q6_K, seed=rows, ids=ids)


@pytest.mark.parametrize("T", [9, 150])
def test_unequal_strides(T):
    a = _run(512, 256, 4, 2, T, False, M.TYPE_Q6_K, up_pad=2, kinds=(0,), seed=T)
    b = _run(512, 256, 4, 2, T, False, M.TYPE_Q6_K, kinds=(1, 2), seed=T)
    assert rel_l2(a, b) <= 2e-3


@pytest.mark.parametrize("td", [M.TYPE_Q6_K, M.TYPE_Q4_K], ids=["q6_k", "q4_k"])
@pytest.mark.parametrize("fused", [True, False], ids=["fused", "separate"])
@pytest.mark.parametrize("D,I,E,K,T", [(256, 256, 6, 2, 3), (768, 256, 20, 3, 40), (1280, 512, 64, 8, 70), (512, 768, 5, 2, 300)])
def test_router_ids_and_tiled_down(D, I, E, K, T, fused, td):
    rng = np.random.default_rng(D + T)
    f = lambda *s: (rng.standard_normal(s) * 0.03).astype(np.float32)  # noqa: E731
    q = lambda t, a: O.quantize(t, a.reshape(-1, a.shape[-1])).reshape(a.shape[:-1] + (-1,))  # noqa: E731
    gate, up, down = q(M.TYPE_Q6_K, f(E, 2 * I if fused else I, D)), q(M.TYPE_Q6_K, f(E, I, D)), q(td, f(E, D, I))
    rw = f(E, D)
    x = rng.standard_normal((T, D)).astype(np.float32)
    act = M.ACT_GELU_ERF_GP1 if fused else M.ACT_SILU
    dev = [M.to_device(a) for a in (gate, up, down, x, rw)]
    L = M.make_layer(D, E, K, I, dev[4], None, M.tensor(dev[0], M.TYPE_Q6_K, [D, gate.shape[1], E]),
                     None if fused else M.tensor(dev[1], M.TYPE_Q6_K, [D, I, E]), M.tensor(dev[2], td, [I, D, E]), fused, act)
    ctx = M.Context(0)
    ctx.reserve(T, D, I, E, K)
    ctx.set_gemm_threshold(1)
    out, counts = M.DeviceBuffer(4 * T * D), M.DeviceBuffer(4 * E)
    lists = M.Routing()
    lists.counts = counts.addr
    tiled = M.DeviceBuffer(M.tiled_bytes(L.down))
    desc = M.Tensor()
    M.check("mi_moe_tile", ctx.tile(L.down, tiled.addr, desc))
    none = M.Tensor.from_buffer_copy(L.down_tiled)
    got = []
    for kind in (2, 1, 0):
        ctx.set_gemm_tiles(kind)
        for with_tiled in (False, True):
            L.down_tiled = desc if with_tiled else none
            for r in (None, lists):
                M.check("forward", ctx.forward(L, dev[3], T, None, out, r))
                got.append(out.download(np.float32, (T, D)))
    assert ctx.take_all_errors() == (0, 0, 0)
    ctx.close()
    o = dict(D=D, E=E, K=K, I=I, router_w=rw, router_b=None, gate=gate, up=None if fused else up, down=down,
             gate_type=M.TYPE_Q6_K, down_type=td, fused=fused, act=act, gating=M.GATING_SOFTMAX_TOPK)
    ref, dbg = O.moe_forward(o, x, None)
    e = rel_l2(got[0], ref)
    print(f"D={D} I={I} E={E} T={T} fused={fused} down {td}: {e:.2e}", flush=True)
    assert e <= 1e-2 and np.array_equal(counts.download(np.int32, (E,)), dbg["counts"])
    for g in got[1:]:
        assert np.array_equal(g.view(np.uint32), got[0].view(np.uint32))
