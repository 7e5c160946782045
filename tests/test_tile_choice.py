"""Which tiles a launch of the prefill products' tile kernels takes. CPU only: the choice is a function of format and shapes
(qlin_probe_gemm_blocks: 1 = 128 tokens x 64 rows, 3 to 8 = that many times 32 tokens x 128 rows, 0 = not one launch of tiles)."""
import ctypes as C

import pytest

from gemm_amd import qlinear
import synth
from tests.test_routes import ALL

SMALL = 1


def blocks(tid, rows, n_cols, n_tok, have_workspace=0):
    return qlinear.load().qlin_probe_gemm_blocks(tid, len(rows), (C.c_int * len(rows))(*rows), n_cols, n_tok, n_cols, have_workspace)


@pytest.mark.parametrize("tid", ALL, ids=lambda t: synth.TYPE_NAMES[t])
def test_tiles_of_the_tokens_and_rounds_that_there_are(tid):
    """one block of 32 tokens less where it would be padding (77, 180 tokens); fewer where a second round of the chip would be nearly
    empty (12288 rows at 300 tokens: 96 x 2 large tiles, 96 x 2 of five blocks are as many; 6144 at 512: 96 large tiles, 192 of four
    blocks); the tensors of a launch together"""
    iq4 = tid in (synth.GGML_IQ4_NL, synth.GGML_IQ4_XS)
    for rows, n_cols, n_tok, want in [
            ((28672,), 4096, 77, 3), ((14336, 14336), 4096, 77, 3), ((28672,), 4096, 180, 6), ((12288,), 4096, 300, 5),
            ((6144,), 4096, 512, SMALL if iq4 else 4), ((4096, 1024, 1024), 4096, 512, SMALL if iq4 else 4), ((14336, 14336), 4096, 512, 8),
            ((14336,), 4096, 512, 8), ((4096,), 4096, 512, SMALL), ((8192,), 2048, 192, SMALL), ((8192, 8192), 2048, 192, 3),
            ((10240,), 4096, 150, 3), ((2048, 256, 256), 2048, 320, SMALL)]:
        assert blocks(tid, rows, n_cols, n_tok) == want, (rows, n_cols, n_tok)


@pytest.mark.parametrize("tid", ALL, ids=lambda t: synth.TYPE_NAMES[t])
def test_divided_launches_and_what_takes_no_tiles(tid):
    assert blocks(tid, (2000,), 5632, 150, 1) == SMALL and blocks(tid, (2900, 1601, 2000), 5632, 150, 1) == SMALL
    if tid != synth.GGML_Q8_0:
        assert blocks(tid, (2400, 2401), 14336, 400, 1) == 8
    assert blocks(tid, (4096,), 4096, 40) == 0 and blocks(tid, (28672,), 4096, 4096, 1) == 0
