"""Token rows that hold a NaN or an infinity among good ones, through the C
ABI: the bad token's output is NaN throughout, and the other tokens' outputs
are bit for bit those of the call with a finite row in its place.

The grouped GEMV of the 32-value types and F16 on its own row lists (no
routing outputs asked for): no id that it reads may place an address outside
the tables, and no work-group may take slots that the call does not have.

The router on such rows: ids in [0, E), each once per token, the lowest ones
where no logit is a number (as the oracle picks them), and weights of NaN, for
every gating and on every path that ranks (fused decode, the chain with and
without its split router, mi_top_k).
"""
import ctypes as C

import numpy as np
import pytest

import mimoe as M
import pyoracle as O
from test_gpu_shared_gb import _quant

pytestmark = pytest.mark.gpu

B32 = {"q8_0": M.TYPE_Q8_0, "q5_0": M.TYPE_Q5_0, "q4_0": M.TYPE_Q4_0, "f16": M.TYPE_F16}


def _layer(rng, t, D, I, E, K, keep):
    def tab(*shape):
        keep.append(M.to_device(np.ascontiguousarray(_quant(t, (rng.standard_normal(shape) * 0.08).astype(np.float32)))))
        return M.tensor(keep[-1], t, list(shape[::-1]))

    keep.append(M.to_device((rng.standard_normal((E, D)) * 0.1).astype(np.float32)))
    return M.make_layer(D, E, K, I, keep[-1], None, tab(E, I, D), tab(E, I, D), tab(E, D, I), False, M.ACT_SILU)


def _check(run, x, bad):
    """run(rows) -> outputs; rows `bad` of x made NaN / infinite one way after another"""
    good = np.setdiff1d(np.arange(len(x)), bad)
    want = run(x)
    assert np.isfinite(want).all()
    for what in ("nan", "nan row", "inf"):
        y = x.copy()
        if what == "nan":
            y[bad, 3] = np.nan
        elif what == "nan row":
            y[bad] = np.nan
        else:
            y[bad, 5], y[bad, 6] = np.inf, -np.inf
        got = run(y)
        assert np.array_equal(got[good].view(np.uint32), want[good].view(np.uint32)), what
        assert np.isnan(got[bad]).all(), what
    assert np.array_equal(run(x).view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("T,bad", [(1, [0]), (4, [2]), (33, [0, 17, 32])])
@pytest.mark.parametrize("E,K", [(64, 8), (128, 2), (20, 3)])
@pytest.mark.parametrize("t", list(B32.values()), ids=list(B32))
def test_gemv_own_row_lists(t, E, K, T, bad):
    D, I = 128, 64
    rng = np.random.default_rng(E + T)
    keep = []
    L = _layer(rng, t, D, I, E, K, keep)
    x = rng.standard_normal((T, D)).astype(np.float32)
    ctx = M.Context(0)
    ctx.reserve(T, D, I, E, K)
    ctx.set_gemm_threshold(1 << 30)
    norm = M.make_norm(M.NORM_RMS, 1e-6)

    def run(rows, normed):
        xd, out = M.to_device(rows), M.DeviceBuffer(4 * T * D)
        if normed:
            M.check("forward_norm", ctx.forward_norm(L, norm, xd, T, None, out))
        else:
            M.check("forward", ctx.forward(L, xd, T, None, out))
        return out.download(np.float32, (T, D))

    for normed in (False, True):
        _check(lambda rows: run(rows, normed), x, bad)
    ctx.close()


def _routed(ctx, L, rows, D, E, K):
    T = len(rows)
    bufs = dict(logits=M.DeviceBuffer(4 * T * E), sel=M.DeviceBuffer(4 * T * K), weights=M.DeviceBuffer(4 * T * K),
                counts=M.DeviceBuffer(4 * E), perm=M.DeviceBuffer(4 * T * K))
    r = M.Routing()
    for k, v in bufs.items():
        setattr(r, k, C.c_void_p(v.addr))
    xd, out = M.to_device(rows), M.DeviceBuffer(4 * T * D)
    M.check("forward", ctx.forward(L, xd, T, None, out, r))
    sel, w = bufs["sel"].download(np.int32, (T, K)), bufs["weights"].download(np.float32, (T, K))
    assert np.array_equal(bufs["counts"].download(np.int32, (E,)), np.bincount(sel.ravel(), minlength=E))
    assert np.array_equal(bufs["perm"].download(np.int32, (T * K,)), O.dispatch(sel, E)[2])
    return out.download(np.float32, (T, D)), sel, w, bufs["logits"].download(np.float32, (T, E))


GATINGS = {"softmax": M.GATING_SOFTMAX_TOPK, "sigmoid": M.GATING_SIGMOID_BIAS, "softmax_all": M.GATING_SOFTMAX_ALL}


@pytest.mark.parametrize("gating", list(GATINGS.values()), ids=list(GATINGS))
@pytest.mark.parametrize("t,E,K,T,bad", [
    (M.TYPE_Q4_K, 64, 8, 1, [0]), (M.TYPE_Q4_K, 20, 3, 1, [0]),                                         # one token
    (M.TYPE_Q4_K, 64, 8, 5, [1, 4]), (M.TYPE_Q4_K, 20, 3, 6, [0, 5]), (M.TYPE_Q4_K, 128, 4, 2, [1]),   # batched decode
    (M.TYPE_Q4_K, 64, 8, 70, [3, 64]), (M.TYPE_Q4_K, 200, 2, 24, [7]),                                  # the chain
    (M.TYPE_Q8_0, 64, 8, 4, [0]), (M.TYPE_Q8_0, 20, 3, 150, [0, 149])],
    ids=["q4k-e64-t1", "q4k-e20-t1", "q4k-e64-t5", "q4k-e20-t6", "q4k-e128-t2", "q4k-e64-t70", "q4k-e200-t24", "q8-e64-t4", "q8-e20-t150"])
def test_router_ids(t, E, K, T, bad, gating):
    D, I = 256, 256
    rng = np.random.default_rng(E + T)
    keep = []
    L = _layer(rng, t, D, I, E, K, keep)
    L.gating = gating
    if gating == M.GATING_SIGMOID_BIAS:
        keep.append(M.to_device((rng.standard_normal(E) * 0.05).astype(np.float32)))
        L.sel_bias, L.routed_scaling, L.gate_eps = keep[-1].addr, 2.5, 1e-20
    if gating == M.GATING_SOFTMAX_ALL:
        keep.append(M.to_device((rng.random(E) + 0.5).astype(np.float32)))
        L.expert_scale = keep[-1].addr
    x = rng.standard_normal((T, D)).astype(np.float32)
    ctx = M.Context(0)
    ctx.reserve(T, D, I, E, K)

    def run(rows):
        out, sel, w, logits = _routed(ctx, L, rows, D, E, K)
        assert sel.min() >= 0 and sel.max() < E and all(len(set(s)) == K for s in sel)
        none = np.isnan(logits).all(1)
        assert np.array_equal(sel[none], np.tile(np.arange(K, dtype=np.int32), (int(none.sum()), 1)))
        assert np.isnan(w[none]).all() and np.isfinite(w[np.isfinite(logits).all(1)]).all()
        # without routing outputs: the products' own row lists where the call has them
        plain = M.DeviceBuffer(4 * T * D)
        M.check("forward", ctx.forward(L, M.to_device(rows), T, None, plain))
        assert np.array_equal(plain.download(np.float32, (T, D)), out, equal_nan=True)
        return out

    # (a sigmoid turns infinite logits into finite scores: NaN rows only)
    good = np.setdiff1d(np.arange(T), bad)
    want = run(x)
    y = x.copy()
    y[bad, 3] = np.nan
    got = run(y)
    assert np.array_equal(got[good].view(np.uint32), want[good].view(np.uint32)) and np.isnan(got[bad]).all()
    if gating == M.GATING_SOFTMAX_TOPK:
        _check(run, x, bad)
    assert ctx.take_errors() == (0, 0)
    ctx.close()


@pytest.mark.parametrize("T", [1, 5, 70])
@pytest.mark.parametrize("E,K,numbers", [(64, 8, 60), (64, 8, 8), (64, 8, 3), (20, 3, 2), (200, 4, 1)])
def test_experts_without_a_logit(E, K, numbers, T):
    """NaN logits of some experts rank behind the numbers, in the order of the ids: with at least K numbers left
    ids, weights and outputs are those without the other experts; with fewer the token is NaN"""
    D, I = 256, 256
    rng = np.random.default_rng(E + numbers)
    keep = []
    L = _layer(rng, M.TYPE_Q4_K, D, I, E, K, keep)
    bias = np.full(E, np.nan, np.float32)
    bias[rng.permutation(E)[:numbers]] = 0.0
    keep.append(M.to_device(bias))
    L.router_b = keep[-1].addr
    ctx = M.Context(0)
    ctx.reserve(T, D, I, E, K)
    out, sel, w, logits = _routed(ctx, L, rng.standard_normal((T, D)).astype(np.float32), D, E, K)
    assert np.array_equal(np.isnan(logits), np.broadcast_to(np.isnan(bias), logits.shape))
    key = np.where(np.isnan(logits), np.inf, -logits)
    assert np.array_equal(sel, np.argsort(key, axis=1, kind="stable")[:, :K])
    whole = numbers >= K
    assert np.isfinite(w).all() == whole and np.isfinite(out).all() == whole
    if whole:
        assert np.allclose(w, O.softmax_selected(np.where(np.isnan(logits), -3e38, logits).astype(np.float32), sel), rtol=1e-6)
    else:
        assert np.isnan(w).all() and np.isnan(out).all()
    ctx.close()


@pytest.mark.parametrize("E,k", [(64, 8), (20, 20), (256, 64), (1, 1), (65, 3)])
def test_top_k_without_numbers(E, k):
    a = np.random.default_rng(E).standard_normal((5, E)).astype(np.float32)
    a[1] = np.nan
    a[3] = -np.inf
    ad, out = M.to_device(a), M.DeviceBuffer(4 * 5 * k)
    ctx = M.Context(0)
    M.check("top_k", ctx.top_k(M.tensor(ad, M.TYPE_F32, [E, 5]), k, M.tensor(out, M.TYPE_I32, [k, 5])))
    assert np.array_equal(out.download(np.int32, (5, k)), O.top_k(a, k))
    ctx.close()
