"""Which kernel qlin_gemm_bf16_any_dev and qlin_gemm_f32_any_dev choose, at both sides of every limit of the few-token kernel
and of the fp32 product on codes. CPU only: the choice is a function of format and shape (qlin_probe_gemm_route: 0 matvec or
decode + dense, 1 and 2 the tile kernels, 3 few tokens; qlin_probe_gemm_f32_route: 1 the product on codes)."""
import pytest

from gemm_amd import qlinear
import synth

ALL = (synth.GGML_Q4_K, synth.GGML_Q5_K, synth.GGML_Q6_K, synth.GGML_Q2_K, synth.GGML_Q3_K, synth.GGML_Q8_0, synth.GGML_Q4_0,
       synth.GGML_IQ4_NL, synth.GGML_IQ4_XS)
FEW, MATVEC = 3, 0


def route(tid, n_rows, n_cols, n_tok, have_workspace=1):
    return qlinear.load().qlin_probe_gemm_route(tid, n_rows, n_cols, n_tok, n_cols, have_workspace)


@pytest.mark.parametrize("tid", ALL, ids=lambda t: synth.TYPE_NAMES[t])
def test_rounded_weights_go_to_the_faster_of_the_few_token_and_tile_kernels(tid):
    q8 = tid == synth.GGML_Q8_0
    for n_rows, n_cols, n_tok, few in [
            (8192, 2048, 64, True), (8193, 2048, 64, q8), (8193, 2048, 48, True), (14336, 4096, 64, True), (14336, 3840, 64, q8),
            (25472, 2048, 64, q8), (25473, 2048, 64, True), (32000, 512, 64, True), (32000, 1536, 64, q8), (48000, 1792, 64, True),
            (19200, 1024, 64, True), (19184, 1024, 64, q8),
            (5120, 2048, 80, True), (5121, 2048, 80, False), (5120, 2048, 128, not q8), (5120, 4096, 128, True), (4096, 2048, 128, True),
            (5120, 1536, 128, False), (4096, 1536, 128, True), (5120, 512, 80, True), (5120, 512, 81, False), (4096, 512, 96, True),
            (4096, 512, 97, q8), (64, 256, 48, True), (64, 256, 49, False), (64, 4096, 129, False)]:
        assert (route(tid, n_rows, n_cols, n_tok) == FEW) == few, (n_rows, n_cols, n_tok)


@pytest.mark.parametrize("tid", ALL, ids=lambda t: synth.TYPE_NAMES[t])
def test_unrounded_tokens_stay_unrounded(tid):
    """whatever the shape: a tile kernel would round their weights"""
    n = 32 if tid == synth.GGML_Q4_K else 4 if tid in (synth.GGML_Q4_0, synth.GGML_IQ4_NL, synth.GGML_IQ4_XS) else 24
    for n_rows, n_cols in [(16, 256), (50000, 256), (50000, 4096), (300, 16384)]:
        assert route(tid, n_rows, n_cols, n) == FEW


@pytest.mark.parametrize("tid,n_rows,n_cols,n_tok,matvec", [
    (synth.GGML_IQ4_NL, 4096, 4096, 1, False), (synth.GGML_IQ4_NL, 8192, 4096, 1, True), (synth.GGML_IQ4_NL, 8192, 4096, 2, False),
    (synth.GGML_IQ4_NL, 40000, 1024, 1, False), (synth.GGML_IQ4_XS, 64, 12288, 1, True), (synth.GGML_IQ4_XS, 64, 12032, 1, False),
    (synth.GGML_IQ3_S, 4607, 4096, 1, False), (synth.GGML_IQ3_S, 4608, 4096, 1, True), (synth.GGML_IQ3_S, 8192, 2048, 1, False),
    (synth.GGML_Q4_0, 16384, 4096, 1, False), (synth.GGML_Q4_0, 16385, 4096, 1, True),
    (synth.GGML_IQ2_XXS, 64, 2816, 1, False), (synth.GGML_IQ2_XXS, 64, 3072, 1, True), (synth.GGML_IQ2_XXS, 4608, 2048, 1, True),
    (synth.GGML_IQ2_XXS, 4096, 4096, 2, False), (synth.GGML_IQ2_XXS, 8193, 4096, 2, True), (synth.GGML_IQ2_XXS, 64, 12288, 2, True),
    (synth.GGML_IQ2_XXS, 8192, 14336, 3, False), (synth.GGML_IQ2_XXS, 8193, 14336, 3, True), (synth.GGML_IQ2_XXS, 8193, 14336, 4, False),
    (synth.GGML_Q4_K, 151936, 4096, 1, False), (synth.GGML_Q8_0, 151936, 4096, 1, False)])
def test_single_tokens_of_large_tensors_go_to_the_matvec(tid, n_rows, n_cols, n_tok, matvec):
    assert route(tid, n_rows, n_cols, n_tok) == (MATVEC if matvec else FEW)
    if tid not in (synth.GGML_IQ3_S, synth.GGML_IQ2_XXS):
        assert route(tid, n_rows, n_cols, n_tok, have_workspace=0) == FEW  # nowhere to widen the activations


@pytest.mark.parametrize("tid", ALL + (synth.GGML_IQ3_S, synth.GGML_IQ2_XXS), ids=lambda t: synth.TYPE_NAMES[t])
def test_fp32_products_that_multiply_codes(tid):
    for n_rows, n_cols, n_tok, codes in [
            (8192, 4096, 7, False), (8192, 4096, 8, True), (8192, 4128, 64, False), (2048, 1024, 32, True), (2047, 1024, 32, False),
            (2304, 1024, 33, True), (2303, 1024, 33, False), (9216, 256, 2000, True)]:
        assert qlinear.load().qlin_probe_gemm_f32_route(tid, n_rows, n_cols, n_tok) == codes, (n_rows, n_cols, n_tok)
    assert not qlinear.load().qlin_probe_gemm_f32_route(synth.GGML_Q4_1, 8192, 4096, 64)


@pytest.mark.parametrize("tid", ALL, ids=lambda t: synth.TYPE_NAMES[t])
def test_long_rows_on_few_tiles_divide_k_where_there_is_a_workspace(tid):
    """the route then is a tile kernel where one piece would take the few-token kernel; rows of up to 16 super-blocks, 64 tokens and
    a call without a workspace keep theirs"""
    assert route(tid, 4096, 14336, 128) == (FEW if tid == synth.GGML_Q8_0 else 2) and route(tid, 4096, 14336, 128, have_workspace=0) == FEW
    assert route(tid, 4096, 14336, 64) == FEW and route(tid, 4096, 4096, 128) == FEW and route(tid, 1024, 4096, 128) == FEW
    assert tid not in (synth.GGML_Q4_K, synth.GGML_Q6_K) or route(tid, 4096, 14336, 768) == 1


@pytest.mark.parametrize("tid", ALL, ids=lambda t: synth.TYPE_NAMES[t])
def test_the_lines_between_the_kernels_past_48_tokens(tid):
    """how often the chip has to go round: 512 small tiles at a time, 256 large ones"""
    q8, small, large = tid == synth.GGML_Q8_0, 2, 1
    for n_rows, n_cols, n_tok, want in [
            (26624, 2560, 64, FEW if q8 else small), (28672, 4096, 64, FEW if q8 else small), (28672, 4096, 128, large if q8 else small),
            (16384, 2048, 256, small), (16385, 2048, 256, large), (16384, 2048, 129, small), (16385, 2048, 130, large),
            (10880, 2048, 200, small), (41984, 2048, 256, large), (32896, 2048, 256, large if q8 else small)]:
        assert route(tid, n_rows, n_cols, n_tok) == want, (n_rows, n_cols, n_tok)


@pytest.mark.parametrize("tid", ALL, ids=lambda t: synth.TYPE_NAMES[t])
def test_tensors_that_fill_few_rounds_stay_in_tiles_beyond_the_lines_for_large_ones(tid):
    """2048 x 2048 at 640 tokens costs less in tiles than to decode (Q8_0: 11008 x 1024 at 328); 28672 x 4096 at 4096 does not, and neither does
    what is wider, or has fewer rows, than the estimates were measured for; without a workspace there is no choice"""
    small, large, dense = 2, 1, 0
    assert route(tid, 2048, 2048, 640) == small if tid != synth.GGML_Q8_0 else route(tid, 11008, 1024, 328) == large
    for n_rows, n_cols, n_tok, want in [(4096, 4096, 2048, dense if tid in (synth.GGML_Q8_0, synth.GGML_Q6_K) else large),
                                        (14336, 4096, 4096, dense), (28672, 4096, 4096, dense), (4096, 14592, 2048, dense)]:
        assert route(tid, n_rows, n_cols, n_tok) == want, (n_rows, n_cols, n_tok)
    assert route(tid, 28672, 4096, 4096, 0) == large
    if tid in (synth.GGML_Q6_K, synth.GGML_Q8_0, synth.GGML_IQ4_NL, synth.GGML_IQ4_XS):
        assert route(tid, 639, 1024, 1860) == dense and route(tid, 640, 1024, 1860) == small
