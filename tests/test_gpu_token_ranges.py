"""GPU parity of bf16 products of 65 to 700 tokens on both sides of the lines between the few-token, small-tile and large-tile
kernels, one tensor and several in a launch, through the C ABI: against the oracle's weights rounded once to bf16 (relative L2 <=
2e-5, the bar of these kernels, which sum the same products in fp32) and several tensors against one call each, bit for bit."""
import ctypes as C

import numpy as np
import pytest

from gemm_amd import qlinear
import synth
from tests.conftest import rel_l2
from tests.test_gpu_gemm_any import FUSED, references

pytestmark = pytest.mark.gpu


def one(tid, dW, dX, n_rows, n_cols, n_tok, ws):
    dY = qlinear.DevBuf.from_numpy(np.full(n_tok * n_rows, np.nan, np.float32))
    qlinear.gemm_bf16_any_dev(tid, dW, dX, dY, n_rows, n_cols, n_tok, n_cols, n_rows, ws)
    qlinear.sync()
    Y = dY.to_numpy(np.float32, (n_tok, n_rows))
    dY.free()
    return Y


# rows a tile and one past it; tensors that take one kernel, and different ones; 512 small tiles and more, alone and together
@pytest.mark.parametrize("n_tok,rows", [(64, (22400,)), (96, (8193, 16)), (77, (5200, 5130)), (128, (25608,)), (130, (16385, 8210)),
                                        (300, (10881, 10945, 130))])
@pytest.mark.parametrize("tid", FUSED, ids=lambda t: synth.TYPE_NAMES[t])
def test_products(oracle, tid, n_tok, rows):
    n_cols, n = 2304, len(rows)
    Ws = [synth.make_weights(tid, r, n_cols, seed=r + tid) for r in rows]
    Xb = synth.to_bf16_bits(synth.make_activation(n_cols, seed=n_tok + tid, tokens=n_tok))
    dWs, dX = [qlinear.DevBuf.from_numpy(W) for W in Ws], qlinear.DevBuf.from_numpy(Xb)
    dYs = [qlinear.DevBuf.from_numpy(np.full(n_tok * r, np.nan, np.float32)) for r in rows]
    ws = qlinear.DevBuf(max(qlinear.gemm_bf16_any_workspace_bytes(r, n_cols) for r in rows))
    qlinear.check(qlinear.load().qlin_gemm_bf16_multi_dev(tid, n, (C.c_void_p * n)(*[d.ptr for d in dWs]), dX.ptr,
                                                          (C.c_void_p * n)(*[d.ptr for d in dYs]), (C.c_int * n)(*rows), n_cols, n_tok, n_cols,
                                                          (C.c_int * n)(*rows), ws.ptr, ws.nbytes, None))
    qlinear.sync()
    for W, dW, dY, r in zip(Ws, dWs, dYs, rows):
        Y = dY.to_numpy(np.float32, (n_tok, r))
        assert np.array_equal(Y, one(tid, dW, dX, r, n_cols, n_tok, ws))
        some = np.r_[0:min(r, 200), max(0, r - 200):r]
        _, designed = references(oracle, tid, W[some] if W.ndim == 2 else W.reshape(r, -1)[some], Xb, n_cols)
        assert rel_l2(Y[:, some], designed) <= 2e-5
    for b in (*dWs, *dYs, dX, ws):
        b.free()
