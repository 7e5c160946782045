"""Which tiles a launch of the prefill products' tile kernels takes. CPU only: the choice is a function of format and shapes
(qlin_probe_gemm_blocks: 1 = 128 tokens x 64 rows, 3 to 8 = that many times 32 tokens x 128 rows, 0 = not one launch of tiles)."""
import ctypes as C

import pytest

from gemm_amd import qlinear
import synth
from tests.test_routes import ALL, route

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
def test_beyond_what_the_estimates_were_fitted_to(tid):
    """many tokens: 64-row tiles read X twice as often, so that large tiles stay (Q2_K 2320 x 1536 at 8568 116 us, in small ones 154), and
    decode + library is not left for tiles (819 x 1024 at 7370 28 us / 42); short rows and very many rows: the tiles of the class, if others
    are estimated to gain less than 8 % (Q4_K 14892 x 512 at 1540 50 us, in five blocks 61; Q2_K 85460 x 1280 at 104 42.0, in four 44.8)"""
    for rows, n_cols, n_tok in [((2320,), 1536, 8568), ((1188,), 2048, 13199), ((14892,), 512, 1540)]:
        assert blocks(tid, rows, n_cols, n_tok) == 8, (rows, n_cols, n_tok)
    for rows, n_cols, n_tok in [((53, 53), 3072, 3034), ((188, 188), 6400, 3359), ((344,), 1024, 3977)]:  # us: 22 / 24, 54 / 77, 13.4 / 16.6 in large ones
        assert blocks(tid, rows, n_cols, n_tok) == SMALL, (rows, n_cols, n_tok)
    assert route(tid, 819, 1024, 7370) == 0
    if tid in (synth.GGML_Q2_K, synth.GGML_Q3_K, synth.GGML_Q4_0):
        assert route(tid, 30544, 14336, 1236) == 1  # more rows than fitted: decode + library takes 1.9 times as long
    if tid in (synth.GGML_Q4_K, synth.GGML_Q2_K, synth.GGML_Q4_0):
        assert blocks(tid, (85460,), 1280, 104) == SMALL
        assert route(tid, 3048, 512, 1816) == 2  # 128 x 64 tiles, as by the lines (Q2_K 14.1 us, in large ones 16.4)


@pytest.mark.parametrize("tid", ALL, ids=lambda t: synth.TYPE_NAMES[t])
def test_divided_launches_and_what_takes_no_tiles(tid):
    assert blocks(tid, (2000,), 5632, 150, 1) == SMALL and blocks(tid, (2900, 1601, 2000), 5632, 150, 1) == SMALL
    if tid != synth.GGML_Q8_0:
        assert blocks(tid, (2400, 2401), 14336, 400, 1) == 8
    assert blocks(tid, (4096,), 4096, 40) == 0 and blocks(tid, (28672,), 4096, 4096, 1) == 0
