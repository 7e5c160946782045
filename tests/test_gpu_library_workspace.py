"""Products through decode and the vendor library's dense GEMM stay inside the workspace that the caller gives, through the C ABI.
The shapes are ones for which the library's first choice of kernel can need more than the 32 MiB that the documented size holds for
it (36 to 62 MiB, by its version), given that size and more: a region behind the workspace, of the same allocation, keeps its
contents, and the result is right in every part of the tensor (relative L2 <= 2e-5 against weights rounded once to bf16, the bar of the dense route; 1e-5 in fp32).
Run once with the library that this process has and once in a process that has loaded torch, whose own copy of the library takes the
place of the system's."""
import os
import subprocess
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)
from gemm_amd import qlinear
import synth
from tests.conftest import rel_l2
from tests.test_gpu_gemm_any import ALL, references

pytestmark = pytest.mark.gpu
BEHIND = 96 << 20
BF16_SHAPES = [(t, r, c, n, pad, more) for t, r, c, n in (
    (synth.GGML_Q8_0, 35536, 2560, 664), (synth.GGML_BF16, 20336, 1536, 1754), (synth.GGML_Q6_K, 6863, 3840, 2629),
    (synth.GGML_IQ2_XS, 70000, 768, 300)) for pad, more in ((0, 0), (64, 0), (0, 31 << 20), (0, 33 << 20), (64, 40 << 20))]


def tall(tid, n_rows, n_cols, seed):
    """rows that repeat a few hundred (an odd count, so that no tile size lines up with the repeats)"""
    few = synth.make_weights(tid, 331, n_cols, seed=seed)
    return np.ascontiguousarray(np.tile(few, (n_rows // 331 + 1, 1))[:n_rows])


def sample(n_rows):
    return np.unique(np.concatenate([np.linspace(0, n_rows - 1, 600).astype(int), np.arange(n_rows - 256, n_rows)]))


def run(call, tid, W, X, n_rows, n_cols, n_tok, ldy, ws_bytes):
    """-> results; the region behind the workspace has been looked at"""
    fill = np.arange((ws_bytes + BEHIND) // 4, dtype=np.uint32)
    bufs = [qlinear.DevBuf.from_numpy(a) for a in (W, X, fill)] + [qlinear.DevBuf(n_tok * ldy * 4)]
    dW, dX, ws, dY = bufs
    qlinear.check(call(tid, dW.ptr, dX.ptr, dY.ptr, n_rows, n_cols, n_tok, n_cols, ldy, ws.ptr, ws_bytes, None))
    qlinear.sync()
    after = ws.to_numpy(np.uint32, fill.shape)
    Y = dY.to_numpy(np.float32, (n_tok, ldy))
    for b in bufs:
        b.free()
    assert np.array_equal(after[ws_bytes // 4:], fill[ws_bytes // 4:])
    return Y


def check_bf16(oracle, tid, n_rows, n_cols, n_tok, pad, more):
    W = tall(tid, n_rows, n_cols, seed=n_tok)
    Xb = synth.to_bf16_bits(synth.make_activation(n_cols, seed=n_rows, tokens=n_tok))
    Y = run(qlinear.load().qlin_gemm_bf16_any_dev, tid, W, Xb, n_rows, n_cols, n_tok, n_rows + pad,
            qlinear.gemm_bf16_any_workspace_bytes(n_rows, n_cols) + more)
    rows = sample(n_rows)
    _, designed = references(oracle, tid, W[rows], Xb, n_cols)
    got = Y[:, rows]
    assert rel_l2(got, designed) <= 2e-5, ALL[tid]
    worst = np.linalg.norm(got - designed, axis=0) / np.linalg.norm(designed, axis=0)
    assert worst.max() <= 1e-4  # no row of its own is off (a lost share of K is 0.1 and more)


def check_fp32(oracle):
    tid, n_rows, n_cols, n_tok = synth.GGML_F32, 82444, 2816, 144
    W = tall(tid, n_rows, n_cols, seed=4)
    X = synth.make_activation(n_cols, seed=5, tokens=n_tok).astype(np.float32)
    Y = run(qlinear.load().qlin_gemm_f32_any_dev, tid, W, X, n_rows, n_cols, n_tok, n_rows, qlinear.gemm_f32_any_workspace_bytes(n_rows, n_cols))
    rows = sample(n_rows)
    exact = X.astype(np.float64) @ oracle.dequant_matrix(tid, W[rows], n_cols).astype(np.float64).T
    assert rel_l2(Y[:, rows], exact) <= 1e-5


@pytest.mark.parametrize("shape", BF16_SHAPES, ids=lambda s: "%s-%dx%d-%d+%d-%d" % ((ALL[s[0]],) + s[1:]))
def test_bf16_product(oracle, shape):
    check_bf16(oracle, *shape)


def test_fp32_product(oracle):
    check_fp32(oracle)


def test_beside_torch():
    done = subprocess.run([sys.executable, "-u", os.path.abspath(__file__)], cwd=ROOT, timeout=110, capture_output=True, text=True)
    assert done.returncode == 0, done.stdout[-2000:] + done.stderr[-2000:]
    assert done.stdout.count("ok") == len(BF16_SHAPES) + 1


if __name__ == "__main__":
    import torch  # noqa: F401 - before the library is loaded
    from oracle.pyoracle import Oracle
    oracle = Oracle()
    loaded = qlinear.load() and {line.split()[-1] for line in open("/proc/self/maps") if "libhipblaslt" in line}
    assert any("torch" in path for path in loaded), loaded
    for s in BF16_SHAPES:
        check_bf16(oracle, *s)
        print(s, "ok", flush=True)
    check_fp32(oracle)
    print("fp32 ok", flush=True)
