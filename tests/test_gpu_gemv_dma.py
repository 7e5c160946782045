"""GPU parity of the matvec on blocks copied to LDS (gemv_dma.hip) against the CPU oracle, at the sizes where it can go wrong: row
groups of 8 and 16 and their remainders, one to sixteen waves, one to four passes over a row, an image slot used again, several
rounds of workgroups, each call shape. Relative L2 <= 1e-5 like every fp32 matvec path; the error of the paths it replaces is 1e-7
to 6e-7."""
import ctypes as C

import numpy as np
import pytest

from gemm_amd import qlinear
import synth
from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu
TOL = 1e-5
FORMATS = [synth.GGML_Q4_K, synth.GGML_Q5_K, synth.GGML_Q6_K, synth.GGML_Q2_K, synth.GGML_Q3_K, synth.GGML_Q8_0, synth.GGML_Q4_0,
           synth.GGML_IQ4_NL, synth.GGML_IQ4_XS, synth.GGML_IQ3_S, synth.GGML_IQ2_XXS]
IDS = [synth.TYPE_NAMES[t] for t in FORMATS]


def weights(tid, n_rows, n_cols, seed):
    """the rows of a small tensor over and over (row r is row r % 211), so that tall tensors are made quickly"""
    base = synth.make_weights(tid, 211, n_cols, seed=seed)
    return np.ascontiguousarray(np.resize(base.reshape(211, -1), (n_rows, base.size // 211)))


def want_of(oracle, tid, W, x, n_cols):
    w = oracle.gemv_f64(tid, np.ascontiguousarray(W[:211]), x, n_cols)
    return np.resize(w, W.shape[0])


# rows: 1 and 2043 (8 a workgroup, the last one short), 2049 (9), 9000 (36: a third group of 4), 40961 (161), 100003 (391)
# columns: 1, 5, 8 super-blocks; 17 and 22 (two passes, some waves one), 43 (three), 54 and 56 (four)
@pytest.mark.parametrize("n_rows,n_cols", [(1, 256), (2043, 1280), (2049, 2048), (9000, 1024), (40961, 1536), (100003, 256), (13000, 5632),
                                           (14001, 4352), (517, 11008), (4100, 13824), (2111, 14336)])
@pytest.mark.parametrize("tid", FORMATS, ids=IDS)
def test_one_matrix(oracle, tid, n_rows, n_cols):
    W, x = weights(tid, n_rows, n_cols, 3 + tid), synth.make_activation(n_cols, seed=n_cols)
    res = synth.make_activation(n_rows, seed=9)
    dW, dx, dy, dr = (qlinear.DevBuf.from_numpy(a) for a in (W, x, np.zeros(n_rows, np.float32), res))
    qlinear.gemv_dev(tid, dW, dx, dy, n_rows, n_cols)
    qlinear.gemv_add_dev(tid, dW, dx, dr, n_rows, n_cols)
    qlinear.sync()
    want = want_of(oracle, tid, W, x, n_cols)
    got, added = dy.to_numpy(np.float32, (n_rows,)), dr.to_numpy(np.float32, (n_rows,))
    assert rel_l2(got, want) <= TOL and rel_l2(added, want + res) <= TOL
    assert np.allclose(got, want, rtol=3e-4, atol=3e-6 * np.abs(want).max())
    assert np.array_equal(added, res + got)


@pytest.mark.parametrize("n_rows,n_cols", [(1, 1024), (2051, 768), (16391, 2048), (9999, 4352), (6157, 14336)])
@pytest.mark.parametrize("tid", FORMATS, ids=IDS)
def test_gate_and_up(oracle, tid, n_rows, n_cols):
    """eight rows of either matrix in a row group, the last groups short"""
    Wg, Wu = weights(tid, n_rows, n_cols, 5 + tid), weights(tid, n_rows, n_cols, 6 + tid)
    x = synth.make_activation(n_cols, seed=7) * np.float32(0.05)
    dg, du, dx, dy = (qlinear.DevBuf.from_numpy(a) for a in (Wg, Wu, x, np.zeros(n_rows, np.float32)))
    qlinear.gemv_silu_mul_dev(tid, dg, du, dx, dy, n_rows, n_cols)
    qlinear.sync()
    g, u = (want_of(oracle, tid, W, x, n_cols).astype(np.float64) for W in (Wg, Wu))
    want = g / (1.0 + np.exp(-g)) * u
    got = dy.to_numpy(np.float32, (n_rows,))
    assert rel_l2(got, want) <= TOL
    assert np.allclose(got, want, rtol=3e-4, atol=3e-6 * np.abs(want).max())


# whole row groups (this kernel); a matrix that ends inside one (another); a group boundary between workgroups
@pytest.mark.parametrize("rows,n_cols", [((2048, 256, 256), 2048), ((16384, 4096), 1024), ((48, 16, 7), 5632), ((50, 16, 16), 2560)])
@pytest.mark.parametrize("tid", FORMATS, ids=IDS)
def test_several_matrices(oracle, tid, rows, n_cols):
    Ws, x = [weights(tid, r, n_cols, 8 + i + tid) for i, r in enumerate(rows)], synth.make_activation(n_cols, seed=2)
    dWs, dx = [qlinear.DevBuf.from_numpy(W) for W in Ws], qlinear.DevBuf.from_numpy(x)
    dys = [qlinear.DevBuf.from_numpy(np.full(r, 7.0, np.float32)) for r in rows]
    qlinear.gemv_multi_dev(tid, dWs, dys, list(rows), dx, n_cols)
    qlinear.sync()
    for W, d, r in zip(Ws, dys, rows):
        assert rel_l2(d.to_numpy(np.float32, (r,)), want_of(oracle, tid, W, x, n_cols)) <= TOL


@pytest.mark.parametrize("tid", FORMATS, ids=IDS)
def test_x_that_is_not_finite_and_zero(oracle, tid):
    n_rows, n_cols = 16400, 1024
    W, x = weights(tid, n_rows, n_cols, 4), synth.make_activation(n_cols, seed=1)
    dW, dy = qlinear.DevBuf.from_numpy(W), qlinear.DevBuf(n_rows * 4)
    for bad in (np.nan, np.inf, -np.inf):
        x[700] = bad
        qlinear.gemv_dev(tid, dW, qlinear.DevBuf.from_numpy(x), dy, n_rows, n_cols)
        qlinear.sync()
        assert np.isnan(dy.to_numpy(np.float32, (n_rows,))).all()
    qlinear.gemv_dev(tid, dW, qlinear.DevBuf.from_numpy(np.zeros(n_cols, np.float32)), dy, n_rows, n_cols)
    qlinear.sync()
    assert not dy.to_numpy(np.float32, (n_rows,)).any()


# That the tests below reach this kernel: qlin_probe_gemv_lds gives waves + 100 x rounds of workgroups.
EVERYWHERE = [synth.GGML_Q5_K, synth.GGML_Q6_K, synth.GGML_Q3_K]
ALL_BUT_GRIDS = EVERYWHERE + [synth.GGML_Q8_0, synth.GGML_Q4_0, synth.GGML_IQ4_NL, synth.GGML_IQ4_XS, synth.GGML_Q2_K]


def route(tid, rows, n_cols, pair=0):
    return qlinear.load().qlin_probe_gemv_lds(tid, pair, len(rows), (C.c_int * len(rows))(*rows), n_cols)


def cases(shapes):
    """(format, shape..., route) of every shape's formats"""
    return [pytest.param(t, *s[1:], id="%s-%s" % (synth.TYPE_NAMES[t], "-".join(map(str, s[1:-1])))) for s in shapes for t in s[0]]


# one pass over a row with nine to sixteen waves: row groups of 8 (the last one short) and of 16; two rounds of workgroups
@pytest.mark.parametrize("tid,n_rows,n_cols,want", cases([
    (EVERYWHERE + [synth.GGML_Q8_0, synth.GGML_IQ3_S], 1030, 2304, 109), (EVERYWHERE + [synth.GGML_Q8_0, synth.GGML_IQ3_S], 2050, 2560, 110),
    (ALL_BUT_GRIDS + [synth.GGML_IQ3_S], 10007, 3840, 115), (ALL_BUT_GRIDS + [synth.GGML_IQ3_S], 14341, 4096, 116),
    ([synth.GGML_IQ2_XXS], 14341, 3072, 112), ([synth.GGML_Q6_K], 86503, 4096, 216)]))
def test_one_matrix_nine_to_sixteen_waves(oracle, tid, n_rows, n_cols, want):
    assert route(tid, [n_rows], n_cols) == want
    test_one_matrix(oracle, tid, n_rows, n_cols)


@pytest.mark.parametrize("tid,n_rows,n_cols,want", cases([
    (EVERYWHERE + [synth.GGML_Q8_0], 1029, 2304, 109), (EVERYWHERE + [synth.GGML_Q8_0], 7001, 3840, 115),
    (ALL_BUT_GRIDS, 2049, 4096, 116), ([synth.GGML_IQ3_S], 7001, 4096, 116), ([synth.GGML_IQ2_XXS], 10001, 2816, 111),
    ([synth.GGML_Q4_K], 9001, 4352, 116), ([synth.GGML_Q6_K], 43507, 4096, 216), ([synth.GGML_Q8_0], 33003, 4352, 214)]))
def test_gate_and_up_nine_to_sixteen_waves(oracle, tid, n_rows, n_cols, want):
    assert route(tid, [n_rows] * 2, n_cols, pair=1) == want
    test_gate_and_up(oracle, tid, n_rows, n_cols)


@pytest.mark.parametrize("tid,rows,n_cols,want", cases([
    (EVERYWHERE + [synth.GGML_Q8_0, synth.GGML_IQ3_S], (1024, 512, 519), 2304, 109), (ALL_BUT_GRIDS, (4096, 1024, 1025), 4096, 116),
    (ALL_BUT_GRIDS + [synth.GGML_IQ3_S], (10240, 48, 17), 3840, 115)]))
def test_several_matrices_nine_to_sixteen_waves(oracle, tid, rows, n_cols, want):
    assert route(tid, rows, n_cols) == want
    test_several_matrices(oracle, tid, rows, n_cols)
