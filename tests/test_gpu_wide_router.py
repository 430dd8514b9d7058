"""Router rows wider than 2048 values (33 chunks of 64 and more: the chunk
partials are added group by group, 32 at a time) through the C ABI: logits bit
for bit the CPU oracle's, ids equal, on the one-launch router and on the
small-batch split over chunks, with widths at the edges of a group, a partial
last chunk, a width no 16-byte load fits, a misaligned x, and experts that are
no multiple of the 16-expert tile; and a k-quant layer whose Q8_K of x comes
from the same launch.
"""
import ctypes as C

import numpy as np
import pytest

import mimoe as M
import pyoracle as O
import workloads as W
from _util import oracle_layer_dict, rel_l2

pytestmark = pytest.mark.gpu


def _layer(D, E, K, I, rng):
    """F16 experts that do not matter here (zeros) behind a seeded router"""
    Wr = (rng.standard_normal((E, D)) * 0.05).astype(np.float32)
    keep = [M.to_device(Wr)] + [M.DeviceBuffer(2 * E * I * D).zero() for _ in range(3)]
    t = [M.tensor(keep[1], M.TYPE_F16, [D, I, E]), M.tensor(keep[2], M.TYPE_F16, [D, I, E]),
         M.tensor(keep[3], M.TYPE_F16, [I, D, E])]
    return M.make_layer(D, E, K, I, keep[0], None, t[0], t[1], t[2], False, M.ACT_SILU), Wr


CASES = [(2080, 20, 40), (2112, 128, 1), (2688, 128, 17), (2816, 128, 200), (4096, 64, 33), (4160, 130, 5),
         (8224, 16, 70)]


@pytest.mark.parametrize("shift", [0, 4], ids=["aligned", "shifted"])
@pytest.mark.parametrize("D,E,T", CASES, ids=[f"D{d}-E{e}-T{t}" for d, e, t in CASES])
def test_wide_router(D, E, T, shift):
    rng = np.random.default_rng(D + E + T)
    K, I = 4, 32
    L, Wr = _layer(D, E, K, I, rng)
    x = rng.standard_normal((T, D)).astype(np.float32)
    xd = M.DeviceBuffer(x.nbytes + 16).upload(x, shift)
    ctx = M.Context(0)
    ctx.reserve(T, D, I, E, K)
    out, lg, sel = M.DeviceBuffer(4 * T * D), M.DeviceBuffer(4 * T * E), M.DeviceBuffer(4 * T * K)
    r = M.Routing()
    r.logits, r.sel = C.c_void_p(lg.addr), C.c_void_p(sel.addr)
    M.check("forward", ctx.forward(L, xd.addr + shift, T, None, out, r))
    ref = O.router_logits(Wr, None, x)
    got = lg.download(np.float32, (T, E))
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))
    assert np.array_equal(sel.download(np.int32, (T, K)), np.argsort(-ref, axis=1, kind="stable")[:, :K])
    ctx.close()


@pytest.mark.parametrize("T", [3, 40])
def test_wide_k_quant_layer(T):
    spec = W.LayerSpec("wide", 4096, 8, 2, 256, True, M.TYPE_Q4_K, M.TYPE_Q6_K, M.ACT_GELU_TANH, "none", 0x5EED0C00)
    ctx = M.Context(0)
    ctx.reserve(T, spec.D, spec.I, spec.E, spec.K)
    g = W.GpuLayer(ctx, spec)
    x = W.gen_x(ctx, spec, T)
    out = M.DeviceBuffer(4 * T * spec.D)
    M.check("forward", ctx.forward(g.layer, x, T, None, out))
    ref, _ = O.moe_forward(oracle_layer_dict(g.download_tables(), spec, g.download_router(), None),
                           x.download(np.float32, (T, spec.D)))
    assert rel_l2(out.download(np.float32, (T, spec.D)), ref) <= 1e-2
    ctx.close()
