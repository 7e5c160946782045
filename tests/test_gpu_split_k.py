"""GPU parity of bf16 products whose K is divided over workgroups (long rows on few tiles, given a workspace), through the C ABI:
against the oracle's weights rounded once to bf16 (relative L2 <= 2e-5, the bar of the tile kernels, which compute the same sums in
one piece), against the same call without a workspace, and several tensors against one call each, bit for bit."""
import ctypes as C

import numpy as np
import pytest

from gemm_amd import qlinear
import synth
from tests.conftest import rel_l2
from tests.test_gpu_gemm_any import ALL, FUSED, references

pytestmark = pytest.mark.gpu
LARGE, SMALL = 1, 2


def product(tid, dW, dX, n_rows, n_cols, n_tok, ldx, ldy, ws):
    dY = qlinear.DevBuf.from_numpy(np.full((n_tok, ldy), -3.0, np.float32))
    qlinear.gemm_bf16_any_dev(tid, dW, dX, dY, n_rows, n_cols, n_tok, ldx, ldy, ws)
    qlinear.sync()
    Y = dY.to_numpy(np.float32, (n_tok, ldy))
    dY.free()
    return Y


# rows: a last tile of 2, of 40, of 93 rows; rows and pitches of Y that allow 16-byte stores of the sums and that do not; K in
# unequal parts (56, 22, 43 super-blocks); tokens: one tile of 77, two (150), three large ones
SHAPES = [(77, 130, 14336, 133, SMALL), (150, 1000, 5632, 1000, SMALL), (260, 1030, 11008, 1032, SMALL)]
BIG = (700, 1501, 14336, 1501, LARGE)


@pytest.mark.parametrize("tid,n_tok,n_rows,n_cols,ldy,tile", [(t,) + s for t in FUSED for s in SHAPES] +
                         [(t,) + BIG for t in (synth.GGML_Q4_K, synth.GGML_Q6_K)])
def test_against_rounded_weights(oracle, tid, n_tok, n_rows, n_cols, ldy, tile):
    route = qlinear.load().qlin_probe_gemm_route(tid, n_rows, n_cols, n_tok, n_cols + 8, 1)
    if tid == synth.GGML_Q4_K:
        assert route == tile
    W = synth.make_weights(tid, n_rows, n_cols, seed=n_rows + tid)
    Xb = synth.to_bf16_bits(synth.make_activation(n_cols, seed=n_tok + tid, tokens=n_tok))
    ldx = n_cols + 8
    Xpad = np.zeros((n_tok, ldx), np.uint16)
    Xpad[:, :n_cols] = Xb
    dW, dX = qlinear.DevBuf.from_numpy(W), qlinear.DevBuf.from_numpy(Xpad)
    ws = qlinear.DevBuf.from_numpy(np.full(qlinear.gemm_bf16_any_workspace_bytes(n_rows, n_cols) // 4, np.nan, np.float32))
    Y = product(tid, dW, dX, n_rows, n_cols, n_tok, ldx, ldy, ws)
    again = product(tid, dW, dX, n_rows, n_cols, n_tok, ldx, ldy, ws)
    whole = product(tid, dW, dX, n_rows, n_cols, n_tok, ldx, ldy, None)
    assert np.array_equal(Y, again)
    assert np.all(Y[:, n_rows:] == -3.0)  # the gap between two tokens' results
    _, designed = references(oracle, tid, W, Xb, n_cols)
    assert rel_l2(Y[:, :n_rows], designed) <= 2e-5
    assert rel_l2(Y[:, :n_rows], whole[:, :n_rows]) <= 2e-6  # the order of the fp32 sums


@pytest.mark.parametrize("tid", [synth.GGML_Q4_K, synth.GGML_Q6_K])
def test_several_tensors_are_one_call_each(tid):
    n_tok, n_cols, rows = 77, 14336, (130, 64, 514)
    dWs = [qlinear.DevBuf.from_numpy(synth.make_weights(tid, r, n_cols, seed=r)) for r in rows]
    dX = qlinear.DevBuf.from_numpy(synth.to_bf16_bits(synth.make_activation(n_cols, seed=3, tokens=n_tok)))
    ws = qlinear.DevBuf(max(qlinear.gemm_bf16_any_workspace_bytes(r, n_cols) for r in rows))
    dYs = [qlinear.DevBuf(n_tok * r * 4) for r in rows]
    qlinear.gemm_bf16_multi_dev(tid, dWs, dX, dYs, list(rows), n_cols, n_tok, n_cols, list(rows), ws)
    qlinear.sync()
    for dW, dY, r in zip(dWs, dYs, rows):
        assert np.array_equal(dY.to_numpy(np.float32, (n_tok, r)), product(tid, dW, dX, r, n_cols, n_tok, n_cols, r, ws))


# every one of them divides: 16-byte stores of the sums (2000 and 2400 rows) and single ones, a last tile of 2, 16, 18, 93 and 96 rows, K in equal and in
# unequal parts (56, 22 and 27 super-blocks), both tile kernels
DIVIDED = [(77, 130, 14336, 133, SMALL), (150, 2000, 5632, 2000, SMALL), (200, 2002, 6912, 2005, SMALL), (400, 2400, 14336, 2404, LARGE)]


@pytest.mark.parametrize("tid,n_tok,n_rows,n_cols,ldy,tile", [(t,) + s for t in FUSED for s in DIVIDED] + [(synth.GGML_Q4_K,) + BIG])
def test_divided_products(oracle, tid, n_tok, n_rows, n_cols, ldy, tile):
    assert qlinear.load().qlin_probe_gemm_parts(tid, n_rows, n_cols, n_tok, n_cols + 8) > 1
    assert qlinear.load().qlin_probe_gemm_route(tid, n_rows, n_cols, n_tok, n_cols + 8, 1) == tile
    test_against_rounded_weights(oracle, tid, n_tok, n_rows, n_cols, ldy, tile)


# an undivided tensor among divided ones; rows that allow 16-byte stores of the sums and that do not; the large tiles; tensors whose
# sums do not fit the workspace together (a call each)
SEVERAL = [(t, (2900, 1601, 2000), 5632, 150, SMALL) for t in FUSED]
SEVERAL += [(t, (2400, 2401), 14336, 400, LARGE) for t in FUSED if t != synth.GGML_Q8_0]
SEVERAL += [(synth.GGML_Q4_K, (1600, 1600, 1604), 5632, 256, SMALL), (synth.GGML_Q4_K, (1536, 1536, 1536), 11776, 700, 0)]
# an undivided tensor among divided ones in large tiles, first and in the middle, a last tile of 26 rows
MIXED_LARGE = {synth.GGML_Q6_K: ((1930, 7680, 1920), 9216, 968), synth.GGML_Q8_0: ((12693, 3815, 3815), 7936, 369)}
SEVERAL += [(t, *MIXED_LARGE.get(t, ((4250, 690, 690), 11520, 915)), LARGE) for t in FUSED]


@pytest.mark.parametrize("tid,rows,n_cols,n_tok,want", SEVERAL)
def test_several_divided_tensors_share_a_launch(oracle, tid, rows, n_cols, n_tok, want):
    lib, n = qlinear.load(), len(rows)
    parts = [lib.qlin_probe_gemm_parts(tid, r, n_cols, n_tok, n_cols) for r in rows]
    assert sum(p > 1 for p in parts) >= 2
    assert lib.qlin_probe_gemm_multi_route(tid, n, (C.c_int * n)(*rows), n_cols, n_tok, n_cols, 1) == want
    Ws = [synth.make_weights(tid, r, n_cols, seed=r + i) for i, r in enumerate(rows)]
    Xb = synth.to_bf16_bits(synth.make_activation(n_cols, seed=3, tokens=n_tok))
    dWs, dX = [qlinear.DevBuf.from_numpy(W) for W in Ws], qlinear.DevBuf.from_numpy(Xb)
    ws_bytes, behind = max(qlinear.gemm_bf16_any_workspace_bytes(r, n_cols) for r in rows), 1 << 20
    ws = qlinear.DevBuf.from_numpy(np.full((ws_bytes + behind) // 4, np.nan, np.float32))
    ldys = [r + 4 * i for i, r in enumerate(rows)]
    dYs = [qlinear.DevBuf.from_numpy(np.full((n_tok, ld), -3.0, np.float32)) for ld in ldys]
    P = C.c_void_p * n
    qlinear.check(lib.qlin_gemm_bf16_multi_dev(tid, n, P(*[d.ptr for d in dWs]), dX.ptr, P(*[d.ptr for d in dYs]), (C.c_int * n)(*rows), n_cols,
                                               n_tok, n_cols, (C.c_int * n)(*ldys), ws.ptr, ws_bytes, None))
    qlinear.sync()
    assert np.isnan(ws.to_numpy(np.float32, ((ws_bytes + behind) // 4,))[ws_bytes // 4:]).all()
    for W, dW, dY, r, ld in zip(Ws, dWs, dYs, rows, ldys):
        Y = dY.to_numpy(np.float32, (n_tok, ld))
        assert np.array_equal(Y, product(tid, dW, dX, r, n_cols, n_tok, n_cols, ld, ws))
        some = np.r_[0:40, r - 150:r]
        _, designed = references(oracle, tid, W.reshape(r, -1)[some], Xb, n_cols)
        assert rel_l2(Y[:, some], designed) <= 2e-5
    for b in (*dWs, *dYs, dX, ws):
        b.free()
