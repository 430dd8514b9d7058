"""Token rows that hold a NaN or an infinity among good ones, through the C
ABI: the bad token's output is NaN throughout, and the other tokens' outputs
are bit for bit those of the call with a finite row in its place.

The grouped GEMV of the 32-value types and F16 on its own row lists (no
routing outputs asked for): no id that it reads may place an address outside
the tables, and no work-group may take slots that the call does not have.
"""
import numpy as np
import pytest

import mimoe as M
from test_gpu_shared_gb import _quant

pytestmark = pytest.mark.gpu

B32 = {"q8_0": M.TYPE_Q8_0, "q5_0": M.TYPE_Q5_0, "q4_0": M.TYPE_Q4_0, "f16": M.TYPE_F16}


def _layer(rng, t, D, I, E, K, keep):
    def tab(*shape):
        keep.append(M.to_device(np.ascontiguousarray(_quant(t, (rng.standard_normal(shape) * 0.08).astype(np.float32)).reshape(shape[:-1] + (-1,)))))
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
