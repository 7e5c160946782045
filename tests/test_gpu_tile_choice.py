"""GPU parity of the public calls in every shape of tile that they choose, through the C ABI: the bits of the 128-token x 64-row kernel called
by name, which is checked against the oracle elsewhere."""
import ctypes as C

import numpy as np
import pytest

from gemm_amd import qlinear
import synth
from tests.test_gpu_gemm_any import ALL, FUSED
from tests.test_tile_choice import blocks

pytestmark = pytest.mark.gpu


# one, two and three tensors; a last tile of 45, 48, 112, 124 and 127 rows; tokens that end a tile early and that fill it
@pytest.mark.parametrize("want,rows,n_cols,n_tok", [(3, (4141, 4144), 1024, 150), (4, (8944,), 1280, 800), (5, (8444, 8447), 1024, 150),
                                                    (5, (16557,), 1024, 150), (6, (8444, 8447), 1024, 180), (8, (8775, 8778), 1024, 250),
                                                    (1, (2048, 256, 256), 2048, 320)])
@pytest.mark.parametrize("tid", FUSED, ids=lambda t: ALL[t])
def test_public_calls_reach_every_tile(tid, want, rows, n_cols, n_tok):
    n = len(rows)
    assert blocks(tid, rows, n_cols, n_tok) == want
    dWs = [qlinear.DevBuf.from_numpy(synth.make_weights(tid, r, n_cols, seed=r + tid)) for r in rows]
    dX = qlinear.DevBuf.from_numpy(synth.to_bf16_bits(synth.make_activation(n_cols, seed=n_tok + tid, tokens=n_tok)))
    dYs = [qlinear.DevBuf.from_numpy(np.full(n_tok * r, np.nan, np.float32)) for r in rows]
    if n == 1:
        qlinear.gemm_bf16_any_dev(tid, dWs[0], dX, dYs[0], rows[0], n_cols, n_tok, n_cols, rows[0], None)
    else:
        P = C.c_void_p * n
        qlinear.check(qlinear.load().qlin_gemm_bf16_multi_dev(tid, n, P(*[d.ptr for d in dWs]), dX.ptr, P(*[d.ptr for d in dYs]),
                                                              (C.c_int * n)(*rows), n_cols, n_tok, n_cols, (C.c_int * n)(*rows), None, 0, None))
    for dW, dY, r in zip(dWs, dYs, rows):
        small = qlinear.DevBuf.from_numpy(np.full(n_tok * r, np.nan, np.float32))
        qlinear.probe_gemm_tile(1, tid, dW, dX, small, r, n_cols, n_tok, n_cols, r)
        qlinear.sync()
        Y = dY.to_numpy(np.float32, (n_tok, r))
        assert np.isfinite(Y).all() and np.array_equal(Y, small.to_numpy(np.float32, (n_tok, r)))
        small.free()
    for b in (*dWs, *dYs, dX):
        b.free()
