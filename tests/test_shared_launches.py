"""Which calls of several tensors (qlin_gemm_bf16_multi_dev) share one launch, and which products divide K. CPU only: the choice is a
function of format and shapes (qlin_probe_gemm_multi_route: 0 a call each, 1 and 2 the tile kernels, 3 few tokens;
qlin_probe_gemm_parts: workgroups that a tile's K is divided over)."""
import ctypes as C

import pytest

from gemm_amd import qlinear
import synth
from tests.test_routes import ALL, route

NAMES = synth.TYPE_NAMES
LARGE, SMALL, FEW = 1, 2, 3


def shared(tid, rows, n_cols, n_tok, have_workspace=1):
    return qlinear.load().qlin_probe_gemm_multi_route(tid, len(rows), (C.c_int * len(rows))(*rows), n_cols, n_tok, n_cols, have_workspace)


def parts(tid, n_rows, n_cols, n_tok):
    return qlinear.load().qlin_probe_gemm_parts(tid, n_rows, n_cols, n_tok, n_cols)


@pytest.mark.parametrize("tid", ALL, ids=lambda t: NAMES[t])
def test_q_k_and_v_share_a_launch(tid):
    for rows, n_cols, n_tok, kernel in [
            ((4096, 1024, 1024), 4096, 128, FEW), ((4096, 1024, 1024), 4096, 256, SMALL), ((5120, 1024, 1024), 5120, 128, FEW),
            ((5120, 1024, 1024), 5120, 256, SMALL), ((8192, 1024, 1024), 8192, 256, SMALL), ((8192, 1024, 1024), 5120, 256, SMALL),
            ((6144, 1024, 1024), 6144, 200, SMALL), ((4096, 2048, 2048), 5376, 256, SMALL), ((8192, 8192, 8192), 8192, 77, SMALL),
            ((6656, 6656, 6656), 6656, 128, SMALL), ((8192, 1024, 1024), 8192, 100, SMALL), ((5376, 5376, 5376), 5376, 100, SMALL)]:
        assert shared(tid, rows, n_cols, n_tok) == kernel, (rows, n_cols, n_tok)
    if tid in (synth.GGML_Q4_K, synth.GGML_Q5_K, synth.GGML_Q3_K):
        for rows, n_cols, n_tok in [((5120, 1024, 1024), 5120, 512), ((8192, 1024, 1024), 8192, 512), ((5120, 1024, 1024), 5120, 1024),
                                    ((6144, 1024, 1024), 6144, 1024)]:
            assert shared(tid, rows, n_cols, n_tok) == SMALL, (rows, n_cols, n_tok)


@pytest.mark.parametrize("tid", ALL, ids=lambda t: NAMES[t])
def test_divided_tensors_share_a_launch(tid):
    """beside an undivided one, and where the workspace holds the parts of all"""
    for rows, n_cols, n_tok in [((8192, 2048, 2048), 8192, 256), ((6144, 1536, 1536), 6144, 200), ((2900, 1601, 2000), 5632, 150)]:
        assert parts(tid, rows[0], n_cols, n_tok) == 1 and parts(tid, rows[1], n_cols, n_tok) > 1
        assert shared(tid, rows, n_cols, n_tok) == SMALL, (rows, n_cols, n_tok)
    rows, n_cols, n_tok = {synth.GGML_Q6_K: ((7680, 1930, 1920), 9216, 968), synth.GGML_Q8_0: ((12693, 3815, 3815), 7936, 369)}.get(
        tid, ((4250, 690, 690), 11520, 915))
    assert [parts(tid, r, n_cols, n_tok) > 1 for r in rows] == [False, True, True] and shared(tid, rows, n_cols, n_tok) == LARGE
    if tid == synth.GGML_Q4_K:  # the sums of three do not fit the workspace
        assert parts(tid, 1536, 11776, 700) == 6 and shared(tid, (1536,) * 3, 11776, 700) == 0 and shared(tid, (1536,) * 2, 11776, 700) == LARGE


@pytest.mark.parametrize("tid", ALL, ids=lambda t: NAMES[t])
def test_a_workspace_takes_no_launch_apart(tid):
    """K and V of up to 1535 rows, whose kernels are Q's without a workspace: dividing their K must not part them from Q (in the few-token
    kernel: from a Q of as many rows as columns)"""
    for n_cols in range(1024, 16385, 1024):
        for kv in (128, 1024, 1535):
            for q in (n_cols * 3 // 4, n_cols, n_cols * 8 // 5):
                for n_tok in range(65, 1025, 29):
                    rows = (q, kv, kv)
                    if q < n_cols and n_tok <= 128:
                        continue
                    if shared(tid, rows, n_cols, n_tok, 0) and all(route(tid, r, n_cols, n_tok) for r in rows):
                        assert shared(tid, rows, n_cols, n_tok), (rows, n_cols, n_tok)


@pytest.mark.parametrize("tid", (synth.GGML_Q4_K, synth.GGML_Q5_K), ids=lambda t: NAMES[t])
def test_gate_and_up_take_the_tiles_that_suit_the_pair(tid):
    """9728 rows at 1024 tokens: 304 large tiles alone are two rounds of the chip, 1216 small ones take less; of the pair, 608 are three
    and 2432 take more. 10880 rows at 200 tokens: 85 large tiles of one tensor and 170 of two are one round, 340 and 680 small ones are
    one and two, and where the two disagree the kernel is the one of 200 large tiles and more"""
    assert shared(tid, (9728, 9728), 2560, 1024) == LARGE and route(tid, 9728, 2560, 1024) == LARGE
    assert shared(tid, (10880, 10880), 2048, 200) == SMALL
    assert shared(tid, (13824, 13824), 5120, 512) == LARGE and shared(tid, (13824, 13824), 5120, 128) == SMALL


@pytest.mark.parametrize("tid", ALL, ids=lambda t: NAMES[t])
def test_down_products_divide_k_and_what_may_share_a_launch_does_not(tid):
    for n_rows, n_cols, n_tok in [(4096, 14336, 256), (2560, 6912, 256), (2048, 5632, 200), (3584, 9728, 200), (1536, 8960, 160), (8192, 8192, 77),
                                  (1024, 8192, 100)]:
        assert parts(tid, n_rows, n_cols, n_tok) > 1, (n_rows, n_cols, n_tok)
    for n_rows, n_cols, n_tok in [(1024, 5120, 128), (5376, 5376, 100), (5440, 5632, 77), (5120, 5120, 256), (1024, 5120, 256), (2048, 5376, 256),
                                  (1024, 8192, 256), (1535, 8192, 256), (1536, 12288, 200), (2048, 4096, 256), (4096, 14336, 64), (4096, 14336, 1025)]:
        assert parts(tid, n_rows, n_cols, n_tok) == 1, (n_rows, n_cols, n_tok)


def test_the_estimates_of_tiles_take_no_division_away():
    """Q6_K past 512 tokens: decode + library by the lines, tiles by the estimates, and faster than either in parts"""
    for n_rows, n_cols, n_tok, n in [(3008, 12032, 630, 3), (2560, 10240, 753, 4), (2432, 9728, 765, 4), (2933, 12288, 599, 3)]:
        assert parts(synth.GGML_Q6_K, n_rows, n_cols, n_tok) == n and route(synth.GGML_Q6_K, n_rows, n_cols, n_tok) == LARGE


def test_large_parts_count_the_padding_of_their_row_tiles():
    """21 row tiles in four parts are 84, which eight dies take as 88: times three token tiles two rounds of 256 compute units"""
    assert parts(synth.GGML_IQ4_NL, 2624, 11520, 612) != 4 or route(synth.GGML_IQ4_NL, 2624, 11520, 612) != LARGE
