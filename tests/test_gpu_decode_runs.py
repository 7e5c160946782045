"""GPU parity of the block decoders where their launches can go wrong: runs of blocks that end inside a workgroup's 512
groups of eight or inside a wave's 64, outputs that are not 16-byte aligned, short and long gathered rows with ids outside
the table. The values are those of the oracle bit for bit; nothing is written behind them."""
import numpy as np
import pytest

from gemm_amd import qlinear
import synth

pytestmark = pytest.mark.gpu
TYPES = list(synth.TYPE_NAMES.items())


def same(got, want):
    assert np.array_equal(np.ascontiguousarray(got).view(np.uint32), np.ascontiguousarray(want, np.float32).view(np.uint32))


@pytest.mark.parametrize("n_rows,blocks", [(1, 1), (3, 5), (5, 13), (1, 129)])
@pytest.mark.parametrize("tid,name", TYPES)
def test_runs_and_rows(oracle, tid, name, n_rows, blocks):
    n_cols = blocks * synth.BLOCK_GEOMETRY[tid][0]
    W = synth.make_weights(tid, n_rows, n_cols, seed=tid + blocks)
    want = oracle.dequant_matrix(tid, W, n_cols)
    n = n_rows * n_cols
    dW = qlinear.DevBuf.from_numpy(W)
    lib = qlinear.load()
    for skip in (0, 1):  # floats in front of the output: aligned to 16 bytes, and to 4 only
        d = qlinear.DevBuf.from_numpy(np.full(n + 8, -5.0, np.float32))
        qlinear.check(lib.qlin_dequant_dev(tid, dW.ptr, d.ptr + 4 * skip, n_rows, n_cols, None))
        qlinear.sync()
        got = d.to_numpy(np.float32, (n + 8,))
        same(got[skip:skip + n].reshape(n_rows, n_cols), want)
        assert np.all(got[:skip] == -5.0) and np.all(got[skip + n:] == -5.0)
        d.free()
    d = qlinear.DevBuf.from_numpy(np.full(n + 8, 7, np.uint16))
    qlinear.dequant_bf16_dev(tid, dW, d, n_rows, n_cols)
    qlinear.sync()
    got = d.to_numpy(np.uint16, (n + 8,))
    assert np.array_equal(got[:n].reshape(n_rows, n_cols), synth.to_bf16_bits(want)) and np.all(got[n:] == 7)
    d.free()
    ids = np.array([n_rows - 1, -1, 0, n_rows, 0, n_rows // 2, n_rows - 1], np.int32)
    dids, d = qlinear.DevBuf.from_numpy(ids), qlinear.DevBuf.from_numpy(np.full(ids.size * n_cols + 8, -5.0, np.float32))
    qlinear.embed_rows_dev(tid, dW, n_rows, dids, ids.size, d, n_cols)
    qlinear.sync()
    got = d.to_numpy(np.float32, (ids.size * n_cols + 8,))
    ok = (ids >= 0) & (ids < n_rows)
    same(got[:-8].reshape(ids.size, n_cols), np.where(ok[:, None], want[np.where(ok, ids, 0)], np.float32(0.0)))
    assert np.all(got[-8:] == -5.0)
    for b in (dW, dids, d):
        b.free()
