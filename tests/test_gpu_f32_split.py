"""GPU parity of the fp32 product on the matrix cores (activations as two fp16 numbers, codes unrounded) at the sizes where
it can go wrong: one and two blocks of 32 tokens and one token past them, ragged row tiles, one super-block and more than
there are parts, K in one part and in several, workspaces that hold only some of the tokens, rows of X at any alignment,
tokens of very different magnitude, magnitudes that differ within a token, infinities and NaN; and one shape just too small
for it. Bar 1e-6: an activation keeps 23 bits (2^-23 = 1.2e-7 of itself at most), the sums are fp32 sums over at most 256
products and 64 super-blocks."""
import numpy as np
import pytest

from gemm_amd import qlinear
import synth
from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu
TYPES = (synth.GGML_Q4_K, synth.GGML_Q5_K, synth.GGML_Q6_K, synth.GGML_Q2_K, synth.GGML_Q3_K, synth.GGML_Q8_0, synth.GGML_Q4_0,
         synth.GGML_IQ4_NL, synth.GGML_IQ4_XS, synth.GGML_IQ3_S, synth.GGML_IQ2_XXS)
NAME = synth.TYPE_NAMES
TOL = 1e-6


def product(tid, W, X, n_rows, n_cols, pad=0, ldy=None):
    n_tok, ldx, ldy = X.shape[0], n_cols + pad, ldy or n_rows
    Xpad = np.full((n_tok, ldx), np.nan, np.float32)  # NaN between the rows: it must not be read into a sum
    Xpad[:, :n_cols] = X
    dW, dX = qlinear.DevBuf.from_numpy(W), qlinear.DevBuf.from_numpy(Xpad)
    dY = qlinear.DevBuf.from_numpy(np.full((n_tok, ldy), -3.0, np.float32))
    ws = qlinear.DevBuf(qlinear.gemm_f32_any_workspace_bytes(n_rows, n_cols))
    qlinear.gemm_f32_any_dev(tid, dW, dX, dY, n_rows, n_cols, n_tok, ldx, ldy, ws)
    qlinear.sync()
    Y = dY.to_numpy(np.float32, (n_tok, ldy))
    for b in (dW, dX, dY, ws):
        b.free()
    assert np.all(Y[:, n_rows:] == -3.0)
    return Y[:, :n_rows]


def takes_codes(tid, n_rows, n_cols, n_tok):
    return qlinear.load().qlin_probe_gemm_f32_route(tid, n_rows, n_cols, n_tok) == 1


def check(oracle, tid, n_tok, n_rows, n_cols, pad=0):
    assert takes_codes(tid, n_rows, n_cols, n_tok) == ((n_tok, n_rows, n_cols) != (64, 2303, 1024))
    W = synth.make_weights(tid, n_rows, n_cols, seed=tid + n_tok + n_rows)
    X = synth.make_activation(n_cols, seed=n_tok + n_cols, tokens=n_tok)
    Y = product(tid, W, X, n_rows, n_cols, pad, n_rows + 3)
    want = X.astype(np.float64) @ oracle.dequant_matrix(tid, W, n_cols).astype(np.float64).T
    assert rel_l2(Y, want) <= TOL, (NAME[tid], n_tok, n_rows, n_cols, rel_l2(Y, want))


@pytest.mark.parametrize("n_tok,n_rows,n_cols,pad", [(8, 8229, 256, 0), (32, 1025, 2304, 4), (33, 3077, 768, 1), (65, 2305, 1024, 6),
                                                     (64, 2303, 1024, 0)])
@pytest.mark.parametrize("tid", TYPES, ids=lambda t: NAME[t])
def test_edges(oracle, tid, n_tok, n_rows, n_cols, pad):
    check(oracle, tid, n_tok, n_rows, n_cols, pad)


@pytest.mark.parametrize("tid", (synth.GGML_Q4_K, synth.GGML_Q6_K), ids=lambda t: NAME[t])
@pytest.mark.parametrize("n_tok,n_rows,n_cols", [(1000, 147, 16384), (64, 16384, 512), (1025, 9300, 256)])
def test_divisions(oracle, tid, n_tok, n_rows, n_cols):
    """tokens in chunks (three quarters of the first shape's workspace hold 460); enough tiles for one part; many token tiles"""
    check(oracle, tid, n_tok, n_rows, n_cols)


@pytest.mark.parametrize("tid", (synth.GGML_Q4_K, synth.GGML_Q6_K, synth.GGML_Q8_0), ids=lambda t: NAME[t])
@pytest.mark.parametrize("n_tok,n_cols", [(9, 2304), (33, 3840), (63, 4096), (384, 4096), (385, 4096), (40, 4352)])
def test_one_launch_and_two_lay_out_the_same(tid, n_tok, n_cols):
    """rows with an odd stride are read singly and laid out by a second launch, aligned ones of up to 4096 elements in the
    first: the product's operand is the same, so its results are, bit for bit"""
    n_rows = 2100
    assert takes_codes(tid, n_rows, n_cols, n_tok)
    W = synth.make_weights(tid, n_rows, n_cols, seed=tid + n_cols)
    X = synth.make_activation(n_cols, seed=n_tok, tokens=n_tok)
    X[n_tok // 2, n_cols - 1] = np.inf
    X[n_tok - 1] *= np.float32(1e-20)
    one, two = (product(tid, W, X, n_rows, n_cols, pad) for pad in (4, 1))
    assert np.array_equal(one, two, equal_nan=True)


@pytest.mark.parametrize("tid", (synth.GGML_Q5_K, synth.GGML_Q8_0, synth.GGML_Q2_K), ids=lambda t: NAME[t])
@pytest.mark.parametrize("n_rows", (4700, 70000))
def test_magnitudes_and_not_finite(oracle, tid, n_rows):
    """each token keeps its own precision whatever its size, up to the largest floats and down to subnormals; one that holds
    an infinity or a NaN gives what the plain sum gives and leaves its neighbours alone (few and many rows: K in parts, in one)"""
    n_cols, n_tok = 512, 40
    W = synth.make_weights(tid, n_rows, n_cols, seed=tid)
    X = synth.make_activation(n_cols, seed=9, tokens=n_tok)
    sizes = {0: 1e30, 1: 1e-30, 2: 3e-42, 3: 65504.0, 4: 0.0, 5: 1e-4, 38: 2e33}
    for t, s in sizes.items():
        X[t] *= np.float32(s)
    X[10, 100], X[11, 7], X[39, 511] = np.inf, np.nan, -np.inf
    Y = product(tid, W, X, n_rows, n_cols)
    at = np.r_[0:50, n_rows - 50:n_rows]
    with np.errstate(invalid="ignore"):
        want = X.astype(np.float64) @ oracle.dequant_matrix(tid, W[at], n_cols).astype(np.float64).T
    Y = Y[:, at]
    for t in range(n_tok):
        if np.all(np.isfinite(X[t])):
            bar = TOL * np.linalg.norm(want[t]) + np.sqrt(len(at)) * 2.0 ** -149  # (a result cannot be finer than a subnormal)
            assert np.linalg.norm(Y[t] - want[t]) <= bar, t
        else:
            assert np.array_equal(np.isnan(Y[t]), np.isnan(want[t])) and np.array_equal(np.isposinf(Y[t]), np.isposinf(want[t])), t


@pytest.mark.parametrize("tid", TYPES, ids=lambda t: NAME[t])
@pytest.mark.parametrize("n_tok,n_rows,n_cols", [(9, 1030, 2304), (33, 24003, 256), (66, 65540, 256)])
def test_tokens_that_are_not_finite(oracle, tid, n_tok, n_rows, n_cols):
    """what the sum over K gives them, wherever and however many their infinities and NaN are, at the ends of the stretches
    of K that are searched together too; K in parts and in one, rows one and four to a thread; neighbours bit for bit as
    without them"""
    W = synth.make_weights(tid, n_rows, n_cols, seed=tid + 1)
    X = synth.make_activation(n_cols, seed=n_tok, tokens=n_tok)
    clean = product(tid, W, X, n_rows, n_cols)
    last = n_cols - 1
    X[0, last] = np.inf
    X[1, [0, last]] = np.inf, np.inf
    X[2, [3, last]] = -np.inf, np.inf
    X[3, :] = np.inf
    X[4, :] = np.nan
    X[5, last // 2:] = -np.inf
    X[7, [min(1023, last), min(1024, last - 1)]] = -np.inf, -np.inf
    X[8, 5] = np.nan
    bad = [0, 1, 2, 3, 4, 5, 7, 8]
    Y = product(tid, W, X, n_rows, n_cols)
    good = np.setdiff1d(np.arange(n_tok), bad)
    assert np.array_equal(Y[good].view(np.uint32), clean[good].view(np.uint32))
    at = np.unique(np.r_[0:60, n_rows // 2:n_rows // 2 + 60, n_rows - 60:n_rows])
    dec = oracle.dequant_matrix(tid, W[at], n_cols).astype(np.float64)
    with np.errstate(invalid="ignore"):
        want = np.stack([(X[t].astype(np.float64) * dec).sum(axis=1) for t in bad])
    got = Y[bad][:, at]
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isposinf(got), np.isposinf(want))
    assert np.array_equal(np.isneginf(got), np.isneginf(want))


@pytest.mark.parametrize("tid", TYPES, ids=lambda t: NAME[t])
@pytest.mark.parametrize("n_tok,n_rows,n_cols", [(9, 8193, 256), (40, 1030, 2304)])
def test_tensor_anywhere_in_its_buffer(oracle, tid, n_tok, n_rows, n_cols):
    """a tensor that starts 2 bytes into a buffer and ends with it: blocks are read from any even address, and the requests
    that a wave makes past its last super-block read nothing"""
    W = synth.make_weights(tid, n_rows, n_cols, seed=tid + n_rows)
    X = synth.make_activation(n_cols, seed=n_tok, tokens=n_tok)
    want = product(tid, W, X, n_rows, n_cols)
    dW = qlinear.DevBuf.from_numpy(np.concatenate([np.zeros(2, np.uint8), W.view(np.uint8).reshape(-1)]))
    dX, dY = qlinear.DevBuf.from_numpy(X), qlinear.DevBuf(n_tok * n_rows * 4)
    ws = qlinear.DevBuf(qlinear.gemm_f32_any_workspace_bytes(n_rows, n_cols))
    qlinear.check(qlinear.load().qlin_gemm_f32_any_dev(tid, dW.ptr + 2, dX.ptr, dY.ptr, n_rows, n_cols, n_tok, n_cols, n_rows, ws.ptr,
                                                       ws.nbytes, None))
    qlinear.sync()
    got = dY.to_numpy(np.float32, (n_tok, n_rows))
    for b in (dW, dX, dY, ws):
        b.free()
    assert np.array_equal(got, want)
    exact = X.astype(np.float64) @ oracle.dequant_matrix(tid, W, n_cols).astype(np.float64).T
    assert rel_l2(got, exact) <= TOL


@pytest.mark.parametrize("n_tok,n_rows,n_cols", [(9, 8229, 256), (40, 1030, 2304)])
@pytest.mark.parametrize("tid", [t for t in TYPES if t not in (synth.GGML_Q4_K, synth.GGML_Q5_K, synth.GGML_Q2_K)], ids=lambda t: NAME[t])
def test_one_hot_activations_return_the_codec_values(oracle, tid, n_tok, n_rows, n_cols):
    """bit for bit where a format subtracts no minimum: code times scales has at most 24 bits, in whatever order"""
    assert takes_codes(tid, n_rows, n_cols, n_tok)
    W = synth.make_weights(tid, n_rows, n_cols, seed=tid)
    ks = ([0, 1, 15, 16, 31, 32, 127, 128, n_cols - 1] + list(range(2, n_cols, 97)))[:n_tok]
    X = np.zeros((n_tok, n_cols), np.float32)
    X[np.arange(len(ks)), ks] = 1.0
    Y = product(tid, W, X, n_rows, n_cols)
    assert np.array_equal(Y[:len(ks)], oracle.dequant_matrix(tid, W, n_cols)[:, ks].T)
    assert not Y[len(ks):].any()


@pytest.mark.parametrize("apart", [10, 15, 22, 30])
@pytest.mark.parametrize("n_rows,n_cols", [(8229, 256), (1030, 2304)])
def test_magnitudes_that_differ_within_a_token(oracle, n_rows, n_cols, apart):
    """one element 2^apart above the others. Rows whose weight of it is not zero are as precise as ever. Rows where it is
    zero show what the others keep: 2^-23 of themselves, and no less than 2^-39 of the largest (half a unit of the second
    fp16 number's subnormals, 2^-25, in a token scaled to [2^14, 2^15))"""
    tid, n_tok, big = synth.GGML_Q8_0, 12, 70
    W = np.ascontiguousarray(synth.make_weights(tid, n_rows, n_cols, seed=apart)).view(np.uint8).reshape(n_rows, -1)
    code = 34 * (big // 32) + 2 + big % 32
    zero = np.arange(n_rows) % 2 == 1
    W[zero, code] = 0
    W[~zero, code] |= 1
    X = synth.make_activation(n_cols, seed=3, tokens=n_tok)
    X[:, big] = np.ldexp(np.abs(X).max(axis=1), apart)
    assert takes_codes(tid, n_rows, n_cols, n_tok)
    Y = product(tid, W, X, n_rows, n_cols)
    dec = oracle.dequant_matrix(tid, W, n_cols).astype(np.float64)
    want = X.astype(np.float64) @ dec.T
    assert rel_l2(Y[:, ~zero], want[:, ~zero]) <= TOL
    kept = np.maximum(2.0 ** -23 * np.abs(X), 2.0 ** -39 * np.abs(X[:, [big]])).astype(np.float64)
    kept[:, big] = 0.0
    small = np.abs(X).astype(np.float64)
    small[:, big] = 0.0
    assert np.all(np.abs(Y - want)[:, zero] <= (kept + TOL * small) @ np.abs(dec[zero]).T)
    if apart <= 15:  # an ordinary outlier: the rows that do not see it keep the bar too
        assert rel_l2(Y[:, zero], want[:, zero]) <= TOL
