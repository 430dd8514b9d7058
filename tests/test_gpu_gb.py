"""The grouped MFMA GEMM of the 32-value types and F16 tables through the C
ABI against the CPU oracle, at the edges of its tiles: 1, 31-33, 63-65 and
127-129 rows per expert and more than one tile of them, widths with an odd
count of 32-value blocks (a half group at the end of a row) and widths no
multiple of a work-group's columns, rows that start at a misaligned even byte
(shifted tables, padded row strides), fused and separate gate/up, relu^2
experts, down tables of another type than gate/up; and mul_mat_id with ids
outside [0, E).  Every case runs on the 32- and on the 128-row tiles, bit for
bit the same.

Bars: the quantized types 1e-2 against the oracle (fp16 operands: 2^-11 per
weight and per activation, and one step of a Q8_0 code, 1 / 127 of a block's
maximum, where a GLU value lies on the edge of two codes); F16 tables 3e-4
(the GLU rows' rounding to fp16, 2^-11 of a value that lies on the edge of two
roundings).
"""
import ctypes as C

import numpy as np
import pytest

import mimoe as M
import pyoracle as O
from _util import rel_l2

pytestmark = pytest.mark.gpu

NAMES = {M.TYPE_Q8_0: "q8_0", M.TYPE_Q5_0: "q5_0", M.TYPE_Q4_0: "q4_0", M.TYPE_F16: "f16"}
TYPES = list(NAMES)
TOL = {t: 1e-2 for t in TYPES}
TOL[M.TYPE_F16] = 3e-4


def _quant(t, w):
    w2 = w.reshape(-1, w.shape[-1])
    return (w2.astype(np.float16).view(np.uint8) if t == M.TYPE_F16 else O.quantize(t, w2)).reshape(w.shape[:-1] + (-1,))


def _device(rows, t, pad, shift, keep):
    """an expert table [E][N][row bytes] with rows `pad` bytes apart more than
    they need and the first row `shift` bytes into its buffer"""
    E, N, rb = rows.shape
    a = np.zeros((E, N, rb + pad), np.uint8)
    a[:, :, :rb] = rows
    buf = M.DeviceBuffer(a.nbytes + 64).upload(a, shift)
    keep.append(buf)
    return buf, [0, rb + pad, (rb + pad) * N, (rb + pad) * N * E]


def _run(t, td, D, I, E, K, counts, fused, act, pad=0, shift=0, seed=0):
    """experts with exactly counts[e] rows through mi_moe_expert_ffn"""
    rng = np.random.default_rng(seed)
    T = sum(counts) // K
    gated = act != M.ACT_RELU_SQR
    f = lambda *s: (rng.standard_normal(s) * 0.05).astype(np.float32)  # noqa: E731
    gate, up, down = _quant(t, f(E, 2 * I if fused else I, D)), _quant(t, f(E, I, D)), _quant(td, f(E, D, I))
    flat = np.concatenate([np.full(n, e, np.int32) for e, n in enumerate(counts)])
    ids = flat.reshape(K, T).T.copy() if K > 1 else flat[rng.permutation(T)].reshape(T, 1)
    x = rng.standard_normal((T, D)).astype(np.float32)
    w = rng.random((T, K)).astype(np.float32) + 0.5
    keep = []

    def tensor(rows, tt, ne):
        buf, nb = _device(rows, tt, pad, shift, keep)
        nb[0] = 2 if tt == M.TYPE_F16 else M.BLOCK_BYTES[tt]
        return M.tensor(buf, tt, ne, nb, offset=shift)

    L = M.make_layer(D, E, K, I, None, None, tensor(gate, t, [D, gate.shape[1], E]),
                     tensor(up, t, [D, I, E]) if gated and not fused else None, tensor(down, td, [I, D, E]), fused, act)
    ctx = M.Context(0)
    ctx.reserve(T, D, I, E, K)
    xd, wd, idd, out = M.to_device(x), M.to_device(w), M.to_device(ids), M.DeviceBuffer(4 * T * D)
    o = dict(D=D, E=E, K=K, I=I, router_w=np.zeros((E, D), np.float32), router_b=None, gate=gate.ravel(),
             up=up.ravel() if gated and not fused else None, down=down.ravel(), gate_type=t, down_type=td, fused=fused, act=act,
             gating=M.GATING_SOFTMAX_TOPK)
    ref, _ = O.moe_forward(o, x, None, sel_in=ids, w_in=w)
    got = {}
    for name, thr, kind in (("gemm", 1, 2), ("gemm128", 1, 1), ("gemm shape", 1, 0), ("gemv", 1 << 30, 0)):
        ctx.set_gemm_threshold(thr)
        ctx.set_gemm_tiles(kind)
        M.check("expert_ffn", ctx.expert_ffn(L, xd, T, None, idd, idd, wd, out))
        got[name] = out.download(np.float32, (T, D))
    for name in ("gemm128", "gemm shape"):   # both tile sizes: the same sums in the same order
        assert np.array_equal(got[name].view(np.uint32), got["gemm"].view(np.uint32)), name
    assert ctx.take_errors() == (0, 0)
    ctx.close()
    e, ev = rel_l2(got["gemm"], ref), rel_l2(got["gemv"], ref)
    print(f"{NAMES[t]}/{NAMES[td]} D={D} I={I} rows {max(counts)} fused={fused} act={act}: gemm {e:.2e} gemv {ev:.2e}", flush=True)
    assert e <= max(TOL[t], TOL[td]) and ev <= 1e-3


@pytest.mark.parametrize("rows", [1, 31, 32, 33, 63, 65, 127, 128, 129, 300])
@pytest.mark.parametrize("t", TYPES, ids=NAMES.values())
def test_tile_rows(t, rows):
    # one expert with `rows` rows, one with one, one with none
    _run(t, t, 128, 64, 3, 1, [rows, 1, 0], True, M.ACT_SILU, seed=rows)


@pytest.mark.parametrize("D,I,rows", [(32, 32, 9), (96, 160, 40), (160, 96, 70), (704, 224, 130), (288, 1056, 20)])
@pytest.mark.parametrize("t", TYPES, ids=NAMES.values())
def test_odd_widths(t, D, I, rows):
    _run(t, t, D, I, 2, 2, [rows, rows], False, M.ACT_GELU_ERF_GP1, seed=D + I)
    _run(t, t, D, I, 2, 2, [rows, rows], False, M.ACT_RELU_SQR, seed=D + I + 1)


@pytest.mark.parametrize("pad,shift", [(0, 2), (2, 0), (6, 2), (4, 4)])
@pytest.mark.parametrize("t", [x for x in TYPES if x != M.TYPE_F16], ids=["q8_0", "q5_0", "q4_0"])
def test_misaligned_rows(t, pad, shift):
    _run(t, t, 160, 96, 3, 2, [50, 40, 34], False, M.ACT_GELU_TANH, pad, shift, seed=pad + shift)
    _run(t, t, 192, 64, 2, 1, [140, 10], True, M.ACT_GELU_ERF, pad, shift, seed=pad + shift + 1)


@pytest.mark.parametrize("t,td", [(M.TYPE_F16, M.TYPE_Q8_0), (M.TYPE_Q4_0, M.TYPE_F16), (M.TYPE_Q5_0, M.TYPE_Q8_0)],
                         ids=["f16-q8_0", "q4_0-f16", "q5_0-q8_0"])
def test_mixed_types(t, td):
    _run(t, td, 224, 96, 3, 2, [45, 33, 90], True, M.ACT_SILU, seed=7)
    _run(t, td, 224, 96, 3, 2, [45, 33, 90], False, M.ACT_RELU_SQR, seed=8)


@pytest.mark.parametrize("t", TYPES, ids=NAMES.values())
def test_mul_mat_id_bad_ids(t):
    rng = np.random.default_rng(3)
    E, N, Kin, n_used, T = 4, 200, 96, 2, 90
    wq = _quant(t, (rng.standard_normal((E, N, Kin)) * 0.05).astype(np.float32))
    b = rng.standard_normal((T, n_used, Kin)).astype(np.float32)
    ids = rng.integers(0, E, (T, n_used)).astype(np.int32)
    bad = ids.copy()
    bad[5, 1], bad[60, 0] = E, -1
    ctx = M.Context(0)
    ctx.reserve(T, Kin, Kin, E, n_used)
    bd, idd, dst = M.to_device(b), M.to_device(bad), M.DeviceBuffer(4 * T * n_used * N)
    wd = M.to_device(wq)
    ref = O.mul_mat_id(t, wq.reshape(E * N, -1), Kin, N, E, b, ids)
    ref[bad != ids] = 0.0
    for kind in (2, 1, 5):   # (5: F16 tables on the 192-row tiles)
        ctx.set_gemm_tiles(kind)
        M.check("mul_mat_id", ctx.mul_mat_id(M.tensor(wd, t, [Kin, N, E]), M.tensor(bd, M.TYPE_F32, [Kin, n_used, T]),
                                             M.tensor(idd, M.TYPE_I32, [n_used, T]), M.tensor(dst, M.TYPE_F32, [N, n_used, T])))
        got = dst.download(np.float32, (T, n_used, N))
        assert not got[bad != ids].any() and rel_l2(got, ref) <= TOL[t]
        assert ctx.take_errors()[0] == 2
    ctx.close()


@pytest.mark.parametrize("rows", [1, 31, 33, 96, 191, 192, 193, 400])
@pytest.mark.parametrize("Kin,N", [(32, 128), (96, 130), (704, 33)])
def test_mul_mat_id_f16_tiles(Kin, N, rows):
    """F16 tables on the 192-row tiles of mul_mat_id (kind 5) against the oracle
    and, bit for bit, the 32- and 128-row tiles: an odd block count, columns no
    multiple of a work-group's, an expert of `rows` rows, one of one, one of none"""
    _mul_mat_id_f16(Kin, N, 3, np.array([0] * rows + [2], np.int32).reshape(-1, 1), (2, 1, 5))


@pytest.mark.parametrize("T", [256, 257, 900])
def test_mul_mat_id_f16_rule(T):
    """above 32 rows per expert the shape rule takes them (16 experts, 16 column groups)"""
    ids = np.random.default_rng(T).permuted(np.tile(np.arange(16, dtype=np.int32), (T, 1)), axis=1)[:, :2].copy()
    _mul_mat_id_f16(96, 2048, 16, ids, (2, 1, 5, 0))


def _mul_mat_id_f16(Kin, N, E, ids, kinds):
    rng = np.random.default_rng(Kin + N)
    T, n_used = ids.shape
    wq = _quant(M.TYPE_F16, (rng.standard_normal((E, N, Kin)) * 0.05).astype(np.float32))
    b = rng.standard_normal((T, 1, Kin)).astype(np.float32)
    ctx = M.Context(0)
    ctx.reserve(T, max(Kin, 32), N, E, n_used)
    ctx.set_gemm_threshold(1)
    wd, bd, idd, dst = M.to_device(wq), M.to_device(b), M.to_device(ids), M.DeviceBuffer(4 * T * n_used * N)
    ref = O.mul_mat_id(M.TYPE_F16, wq.reshape(E * N, -1), Kin, N, E, b, ids)
    got = []
    for kind in kinds:
        ctx.set_gemm_tiles(kind)
        M.check("mul_mat_id", ctx.mul_mat_id(M.tensor(wd, M.TYPE_F16, [Kin, N, E]), M.tensor(bd, M.TYPE_F32, [Kin, 1, T]),
                                             M.tensor(idd, M.TYPE_I32, [n_used, T]), M.tensor(dst, M.TYPE_F32, [N, n_used, T])))
        got.append(dst.download(np.float32, (T, n_used, N)))
    assert rel_l2(got[0], ref) <= 1e-5   # (exact fp16 products, fp32 sums of Kin terms in another order)
    for g in got[1:]:
        assert np.array_equal(g.view(np.uint32), got[0].view(np.uint32))
    ctx.close()


def test_more_rows_than_one_pass_holds():
    """past 983,040 tokens of 2048 values the activation rows outgrow the
    GEMM's 32-bit buffer offsets and the call runs in passes: rows on both
    sides of the seam, bit for bit those of small calls of their own; the
    routing outputs are the whole call's"""
    T, D, I, E, cut = 983_200, 2048, 32, 2, 983_040
    rng = np.random.default_rng(11)
    t = M.TYPE_Q8_0
    tabs = [M.to_device(_quant(t, (rng.standard_normal(s) * 0.05).astype(np.float32)))
            for s in ((E, I, D), (E, I, D), (E, D, I))]
    rw = M.to_device((rng.standard_normal((E, D)) * 0.05).astype(np.float32))
    L = M.make_layer(D, E, 1, I, rw, None, M.tensor(tabs[0], t, [D, I, E]), M.tensor(tabs[1], t, [D, I, E]),
                     M.tensor(tabs[2], t, [I, D, E]), False, M.ACT_SILU)
    ctx = M.Context(0)
    ctx.reserve(T, D, I, E, 1)
    x, out = M.DeviceBuffer(4 * T * D), M.DeviceBuffer(4 * T * D)
    M.check("fill", ctx.fill_normal(x, T * D, 5, 1, 0.0, 1.0))
    counts, sel = M.DeviceBuffer(4 * E), M.DeviceBuffer(4 * T)
    r = M.Routing()
    r.counts, r.sel = C.c_void_p(counts.addr), C.c_void_p(sel.addr)
    M.check("forward", ctx.forward(L, x, T, None, out, r))
    ids = sel.download(np.int32, (T,))
    assert np.array_equal(counts.download(np.int32, (E,)), np.bincount(ids, minlength=E))
    for lo, n in ((0, 100), (cut - 90, 200), (T - 64, 64)):
        small = M.DeviceBuffer(4 * n * D)
        M.check("forward", ctx.forward(L, x.addr + 4 * lo * D, n, None, small))
        assert np.array_equal(small.download(np.uint32, (n, D)), out.download(np.uint32, (n, D), 4 * lo * D))
    assert ctx.take_errors() == (0, 0)
    ctx.close()


@pytest.mark.parametrize("T,n_used", [(1, 1_000_000), (2, 500_000)], ids=["one_token", "two_passes"])
def test_mul_mat_id_rows_past_the_offsets(T, n_used):
    """a token's rows past the GEMM's 32-bit buffer offsets (2.05e9 values: the
    GEMV takes the call), and two tokens that fit only one by one (a pass
    each): rows at both ends and on both sides of the seam against the oracle"""
    t, Kin, N, E = M.TYPE_Q8_0, 2048, 32, 4
    rng = np.random.default_rng(T)
    wq = _quant(t, (rng.standard_normal((E, N, Kin)) * 0.05).astype(np.float32))
    rows = T * n_used
    ids = rng.integers(0, E, (T, n_used)).astype(np.int32)
    ctx = M.Context(0)
    ctx.reserve(rows, Kin, N, E, 1)
    wd, b, idd, dst = M.to_device(wq), M.DeviceBuffer(4 * rows * Kin), M.to_device(ids), M.DeviceBuffer(4 * rows * N)
    M.check("fill", ctx.fill_normal(b, rows * Kin, 7, 1, 0.0, 1.0))
    M.check("mul_mat_id", ctx.mul_mat_id(M.tensor(wd, t, [Kin, N, E]), M.tensor(b, M.TYPE_F32, [Kin, n_used, T]),
                                         M.tensor(idd, M.TYPE_I32, [n_used, T]), M.tensor(dst, M.TYPE_F32, [N, n_used, T])))
    for lo in (0, rows // 2 - 30, rows - 60):
        part = b.download(np.float32, (1, 60, Kin), 4 * lo * Kin)
        ref = O.mul_mat_id(t, wq.reshape(E * N, -1), Kin, N, E, part, ids.ravel()[lo:lo + 60].reshape(1, -1))
        assert rel_l2(dst.download(np.float32, (1, 60, N), 4 * lo * N), ref) <= (1e-4 if T == 1 else TOL[t])
    assert ctx.take_errors() == (0, 0)
    ctx.close()
