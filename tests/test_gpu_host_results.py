"""The host-pointer matvecs store their results over the bus and wait for a flag: many calls of changing shape, each result whole and
the same bits as the first time, the residual added to what the caller has, from one thread and from several."""
import threading

import numpy as np
import pytest

from gemm_amd import qlinear
import synth
from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu
# a kernel of its own for each: copied blocks, Q4_K, a format of neither (results by a copy kernel), ragged dense rows
CASES = [(synth.GGML_Q6_K, 515, 1024), (synth.GGML_Q4_K, 2048, 2048), (synth.GGML_Q4_1, 300, 512), (synth.GGML_BF16, 33, 100),
         (synth.GGML_Q8_0, 1, 256), (synth.GGML_IQ2_XXS, 4096, 512)]


def results(case):
    tid, n_rows, n_cols = case
    W, U = (synth.make_weights(tid, n_rows, n_cols, seed=s) for s in (1, 2))
    x, res = synth.make_activation(n_cols, seed=3) * np.float32(0.05), synth.make_activation(n_rows, seed=4)
    return W, U, x, res


def calls(W, U, x, res, tid, n_cols):
    y = qlinear.matvec(tid, W, x, n_cols)
    return y, qlinear.matvec_add(tid, W, x, n_cols, res.copy()), qlinear.matvec_silu_mul(tid, W, tid, U, x, n_cols)


def test_many_calls(oracle):
    inputs = [results(c) for c in CASES]
    first = [calls(*i, c[0], c[2]) for i, c in zip(inputs, CASES)]
    for (W, U, x, res), (tid, _, n_cols), (y, added, act) in zip(inputs, CASES, first):
        want = oracle.gemv_f64(tid, W, x, n_cols)
        up = oracle.gemv_f64(tid, U, x, n_cols)
        assert rel_l2(y, want) <= 1e-5 and rel_l2(added, want + res) <= 1e-5 and rel_l2(act, want / (1 + np.exp(-want)) * up) <= 1e-5
    for _ in range(60):
        for i, c, f in zip(inputs, CASES, first):
            assert all(np.array_equal(a, b) for a, b in zip(calls(*i, c[0], c[2]), f))


def test_several_threads():
    inputs = [results(c) for c in CASES]
    first = [calls(*i, c[0], c[2]) for i, c in zip(inputs, CASES)]
    wrong = []

    def work(k):
        for n in range(40):
            j = (n + k) % len(CASES)
            if not all(np.array_equal(a, b) for a, b in zip(calls(*inputs[j], CASES[j][0], CASES[j][2]), first[j])):
                wrong.append((k, n))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
