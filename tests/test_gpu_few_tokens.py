"""GPU parity of the few-token product (up to 128 tokens) at the sizes where it can go wrong: every capacity of its
instances and one token past it, fewer super-blocks than waves, an uneven number per wave, ragged last row tiles, one and
two row tiles per workgroup, padded X and Y, several tensors in one launch. Unrounded codes are held to 2e-6 (fp32 sums of
at most 2304 products and their block scales: a few units of 2^-24 each), rounded weights to 2e-5 against weights rounded
once to bf16, as for the tile kernels."""
import numpy as np
import pytest

from gemm_amd import qlinear
import synth
from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu
EXACT_MAX = {synth.GGML_Q4_K: 32, synth.GGML_Q5_K: 24, synth.GGML_Q6_K: 24, synth.GGML_Q2_K: 24, synth.GGML_Q3_K: 24,
             synth.GGML_Q8_0: 24, synth.GGML_Q4_0: 4, synth.GGML_IQ4_NL: 4, synth.GGML_IQ4_XS: 4, synth.GGML_IQ3_S: 4,
             synth.GGML_IQ2_XXS: 4}
NAME = synth.TYPE_NAMES


GRID = (synth.GGML_IQ3_S, synth.GGML_IQ2_XXS)  # up to 64 tokens


def check(oracle, tid, rows_list, n_cols, n_tok, sample=None, pad=8):
    rng = np.random.default_rng(tid * 1000 + n_tok)
    Ws = [synth.make_weights(tid, r, n_cols, seed=tid + 7 * i + n_tok) for i, r in enumerate(rows_list)]
    Xb = synth.to_bf16_bits(synth.make_activation(n_cols, seed=n_tok, tokens=n_tok))
    ldx = n_cols + pad
    Xpad = np.full((n_tok, ldx), 0x7FC0, np.uint16)  # NaN between the rows: it must not be read into a sum
    Xpad[:, :n_cols] = Xb
    dX = qlinear.DevBuf.from_numpy(Xpad)
    dWs = [qlinear.DevBuf.from_numpy(w) for w in Ws]
    ldys = [r + 3 for r in rows_list]
    dYs = [qlinear.DevBuf.from_numpy(np.full((n_tok, ld), -3.0, np.float32)) for ld in ldys]
    ws = qlinear.DevBuf(max(qlinear.gemm_bf16_any_workspace_bytes(r, n_cols) for r in rows_list))
    assert qlinear.load().qlin_probe_gemm_route(tid, rows_list[0], n_cols, n_tok, ldx, 1) == 3
    qlinear.gemm_bf16_multi_dev(tid, dWs, dX, dYs, rows_list, n_cols, n_tok, ldx, ldys, ws)
    qlinear.sync()
    Xf = synth.bf16_bits_to_f32(Xb).astype(np.float64)
    for W, dY, r, ld in zip(Ws, dYs, rows_list, ldys):
        Y = dY.to_numpy(np.float32, (n_tok, ld))
        assert np.all(Y[:, r:] == -3.0)
        at = np.arange(r) if sample is None or r <= 200 else np.unique(np.concatenate([rng.choice(r, sample, replace=False), np.arange(r - 40, r)]))
        dec = oracle.dequant_matrix(tid, W[at], n_cols)
        if n_tok > EXACT_MAX[tid]:
            dec = synth.bf16_bits_to_f32(synth.to_bf16_bits(dec))
        want = Xf @ dec.astype(np.float64).T
        assert rel_l2(Y[:, at], want) <= (2e-5 if n_tok > EXACT_MAX[tid] else 2e-6), (NAME[tid], n_tok, r)
    for b in dWs + dYs + [dX, ws]:
        b.free()


@pytest.mark.parametrize("n_tok", [1, 4, 5, 8, 9, 16, 17, 24, 25, 32, 33, 48, 49, 64, 65, 80, 81, 96, 97, 128])
@pytest.mark.parametrize("tid", sorted(EXACT_MAX), ids=lambda t: NAME[t])
def test_every_capacity(oracle, tid, n_tok):
    if n_tok <= 64 or tid not in GRID:
        check(oracle, tid, [37], 2304, n_tok)  # nine super-blocks over eight waves, three row tiles, the last of five rows


@pytest.mark.parametrize("n_tok", [3, 8, 16, 24, 32, 48, 64])
@pytest.mark.parametrize("tid", sorted(EXACT_MAX), ids=lambda t: NAME[t])
def test_two_row_tiles_per_workgroup(oracle, tid, n_tok):
    rows, n_cols = ([4663], 768) if n_tok % 16 == 0 else ([4627, 130, 33], 256)
    check(oracle, tid, rows, n_cols, n_tok, sample=60)


@pytest.mark.parametrize("n_tok", [65, 81, 97, 128])
@pytest.mark.parametrize("tid", sorted(set(EXACT_MAX) - set(GRID)), ids=lambda t: NAME[t])
def test_two_row_tiles_of_many_tokens(oracle, tid, n_tok):
    check(oracle, tid, [4663], 2048 if n_tok <= 96 else 4096, n_tok, sample=40)


@pytest.mark.parametrize("n_tok,n_cols", [(7, 512), (40, 512), (100, 512), (40, 2048), (90, 2048), (100, 2048)])
@pytest.mark.parametrize("tid", sorted(EXACT_MAX), ids=lambda t: NAME[t])
def test_tensors_of_one_launch_equal_a_call_each(tid, n_tok, n_cols):
    """bit for bit, though the joint launch puts two row tiles in a workgroup and a call of its own one"""
    rows = [2500, 2300, 48]
    Ws = [synth.make_weights(tid, r, n_cols, seed=r) for r in rows]
    dX = qlinear.DevBuf.from_numpy(synth.to_bf16_bits(synth.make_activation(n_cols, seed=3, tokens=n_tok)))
    ws = qlinear.DevBuf(qlinear.gemm_bf16_any_workspace_bytes(max(rows), n_cols))
    dWs, got = [qlinear.DevBuf.from_numpy(w) for w in Ws], []
    for together in (True, False):
        dYs = [qlinear.DevBuf(n_tok * r * 4) for r in rows]
        if together:
            qlinear.gemm_bf16_multi_dev(tid, dWs, dX, dYs, rows, n_cols, n_tok, n_cols, rows, ws)
        else:
            for w, y, r in zip(dWs, dYs, rows):
                qlinear.gemm_bf16_any_dev(tid, w, dX, y, r, n_cols, n_tok, n_cols, r, ws)
        qlinear.sync()
        got.append([y.to_numpy(np.uint32, (n_tok, r)) for y, r in zip(dYs, rows)])
    for a, b in zip(*got):
        assert np.array_equal(a, b)


# K = 1024: four waves with a super-block each, and in it eight sums of 32 exact products that the matrix instruction adds,
# scaled and added in fp32. That is about a dozen roundings of half a unit of 2^-24 at most, of partial sums that grow to
# the result, and their root mean square stays below 1.5 units; a code that goes in with a constant which comes off after a
# rounding shows as more.
UNROUNDED_BAR = 1.75 * 2.0 ** -24


@pytest.mark.parametrize("tid,n_tok", [(t, n) for t in sorted(EXACT_MAX) for n in (3, 8, 16, 24) if n <= EXACT_MAX[t]],
                         ids=str)
def test_unrounded_codes_keep_fp32_precision(oracle, tid, n_tok):
    n_rows, n_cols = 1024, 1024
    W = synth.make_weights(tid, n_rows, n_cols, seed=tid)
    Xb = synth.to_bf16_bits(synth.make_activation(n_cols, seed=n_tok, tokens=n_tok))
    dW, dX, dY = qlinear.DevBuf.from_numpy(W), qlinear.DevBuf.from_numpy(Xb), qlinear.DevBuf(n_tok * n_rows * 4)
    ws = qlinear.DevBuf(qlinear.gemm_bf16_any_workspace_bytes(n_rows, n_cols))
    qlinear.gemm_bf16_any_dev(tid, dW, dX, dY, n_rows, n_cols, n_tok, n_cols, n_rows, ws)
    qlinear.sync()
    Y = dY.to_numpy(np.float32, (n_tok, n_rows))
    for b in (dW, dX, dY, ws):
        b.free()
    want = synth.bf16_bits_to_f32(Xb).astype(np.float64) @ oracle.dequant_matrix(tid, W, n_cols).astype(np.float64).T
    assert rel_l2(Y, want) <= UNROUNDED_BAR, (NAME[tid], n_tok, rel_l2(Y, want) * 2.0 ** 24)


@pytest.mark.parametrize("tid,n_rows,n_cols,n_tok", [
    (synth.GGML_IQ4_NL, 70, 12288, 1), (synth.GGML_IQ4_XS, 70, 12288, 1), (synth.GGML_IQ3_S, 70, 12288, 1), (synth.GGML_IQ2_XXS, 70, 3072, 1),
    (synth.GGML_IQ2_XXS, 4610, 1280, 1), (synth.GGML_IQ2_XXS, 70, 12288, 2)], ids=str)
def test_tokens_that_go_to_the_matvec(oracle, tid, n_rows, n_cols, n_tok):
    """exact weights as in the few-token kernel, rows of X and Y at a distance, nothing written between them"""
    W = synth.make_weights(tid, n_rows, n_cols, seed=tid)
    Xb = synth.to_bf16_bits(synth.make_activation(n_cols, seed=n_tok, tokens=n_tok))
    ldx, ldy = n_cols + 8, n_rows + 3
    Xpad = np.full((n_tok, ldx), 0x7FC0, np.uint16)
    Xpad[:, :n_cols] = Xb
    assert qlinear.load().qlin_probe_gemm_route(tid, n_rows, n_cols, n_tok, ldx, 1) == 0
    dW, dX, dY = qlinear.DevBuf.from_numpy(W), qlinear.DevBuf.from_numpy(Xpad), qlinear.DevBuf.from_numpy(np.full((n_tok, ldy), -3.0, np.float32))
    ws = qlinear.DevBuf(qlinear.gemm_bf16_any_workspace_bytes(n_rows, n_cols))
    qlinear.gemm_bf16_any_dev(tid, dW, dX, dY, n_rows, n_cols, n_tok, ldx, ldy, ws)
    qlinear.sync()
    Y = dY.to_numpy(np.float32, (n_tok, ldy))
    for b in (dW, dX, dY, ws):
        b.free()
    assert np.all(Y[:, n_rows:] == -3.0)
    want = synth.bf16_bits_to_f32(Xb).astype(np.float64) @ oracle.dequant_matrix(tid, W, n_cols).astype(np.float64).T
    assert rel_l2(Y[:, :n_rows], want) <= 2e-6


@pytest.mark.parametrize("n_tok", [3, 8, 16, 24, 40])
@pytest.mark.parametrize("tid", sorted(EXACT_MAX), ids=lambda t: NAME[t])
def test_a_token_that_is_not_finite_leaves_the_others_alone(tid, n_tok):
    """also where two tokens share an operand of zeros and eight-token halves"""
    n_rows, n_cols = 70, 2304
    W = synth.make_weights(tid, n_rows, n_cols, seed=tid)
    Xb = synth.to_bf16_bits(synth.make_activation(n_cols, seed=n_tok, tokens=n_tok))
    bad = np.unique([1, n_tok // 2 + 1, n_tok - 1])
    got = []
    for spoil in (False, True):
        X = Xb.copy()
        if spoil:
            X[bad[0], 5], X[bad[-1], 700], X[bad[0], n_cols - 1] = 0x7F80, 0x7FC0, 0xFF80
        dW, dX, dY = qlinear.DevBuf.from_numpy(W), qlinear.DevBuf.from_numpy(X), qlinear.DevBuf(n_tok * n_rows * 4)
        ws = qlinear.DevBuf(qlinear.gemm_bf16_any_workspace_bytes(n_rows, n_cols))
        qlinear.gemm_bf16_any_dev(tid, dW, dX, dY, n_rows, n_cols, n_tok, n_cols, n_rows, ws)
        qlinear.sync()
        got.append(dY.to_numpy(np.uint32, (n_tok, n_rows)))
        for b in (dW, dX, dY, ws):
            b.free()
    rest = np.setdiff1d(np.arange(n_tok), [bad[0], bad[-1]])
    assert np.array_equal(got[0][rest], got[1][rest])
    spoiled = got[1][[bad[0], bad[-1]]].view(np.float32)
    assert not np.isfinite(spoiled).any()


@pytest.mark.parametrize("rows,n_cols,n_tok", [((70, 33, 5), 3072, 1), ((70, 33), 12288, 2), ((4610, 33), 2048, 1)])
def test_tensors_that_all_go_to_the_matvec(oracle, rows, n_cols, n_tok):
    """what a call per tensor gives, bit for bit, from one widening of X; a tensor that does not go there (the last case's
    second) changes nothing about that"""
    tid, rows = synth.GGML_IQ2_XXS, list(rows)
    Ws = [synth.make_weights(tid, r, n_cols, seed=r) for r in rows]
    ldx = n_cols + 8
    X = np.full((n_tok, ldx), 0x7FC0, np.uint16)
    X[:, :n_cols] = synth.to_bf16_bits(synth.make_activation(n_cols, seed=5, tokens=n_tok))
    ldys = [r + 2 for r in rows]
    dWs, dX = [qlinear.DevBuf.from_numpy(w) for w in Ws], qlinear.DevBuf.from_numpy(X)
    ws = qlinear.DevBuf(qlinear.gemm_bf16_any_workspace_bytes(max(rows), n_cols))
    got = []
    for together in (True, False):
        dYs = [qlinear.DevBuf.from_numpy(np.full((n_tok, ld), -3.0, np.float32)) for ld in ldys]
        if together:
            qlinear.gemm_bf16_multi_dev(tid, dWs, dX, dYs, rows, n_cols, n_tok, ldx, ldys, ws)
        else:
            for w, y, r, ld in zip(dWs, dYs, rows, ldys):
                qlinear.gemm_bf16_any_dev(tid, w, dX, y, r, n_cols, n_tok, ldx, ld, ws)
        qlinear.sync()
        got.append([y.to_numpy(np.float32, (n_tok, ld)) for y, ld in zip(dYs, ldys)])
        for b in dYs:
            b.free()
    for b in dWs + [dX, ws]:
        b.free()
    Xf = synth.bf16_bits_to_f32(X[:, :n_cols]).astype(np.float64)
    for W, a, b, r in zip(Ws, *got, rows):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32)) and np.all(a[:, r:] == -3.0)
        assert rel_l2(a[:, :r], Xf @ oracle.dequant_matrix(tid, W, n_cols).astype(np.float64).T) <= 2e-6
