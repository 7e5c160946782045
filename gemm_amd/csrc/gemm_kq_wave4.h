/*
 * gemm_kq_wave4.h - the fused block-format x bf16 prefill GEMM (Q2_K ... Q6_K, Q8_0, IQ4_NL, IQ4_XS, Q4_0: the formats of
 * gemm_kq_formats.h) in tiles of 128 rows x 256 tokens, or 192, 160, 128, 96: four waves per workgroup, one per SIMD. The kernel and
 * its launch as templates over the format; gemm_kq_wave4_*.hip instantiate them.
 *
 *   Y[t*ldy + r] = sum_k X[t*ldx + k] * decode(W)[r][k]      X bf16, Y fp32, fp32 accumulate
 *
 * The contraction of tf_gemm_f16_mt_tokenmajor (common/transformer.h:4487, generic branch :4535-4572) with the
 * weights decoded as dequantize_row_q4_K / _q5_K / _q6_K / _q8_0 do (common/ggml_dequant.h:1592-1618, :1620-1660,
 * :1662-1700, :1479-1489; y = (d*sc)*q - dmin*m, resp. d*sc*(q - 32), resp. d*q, in fp32) and rounded once to bf16,
 * nearest even. What the reference's
 * fused kernel does per tile for every type (rdna4/dequant/bench_dequant.c:359-459), on this part's terms.
 *
 * What the shape follows from, measured on MI355X with one wave per SIMD (cycles that the matrix pipe waits for
 * an instruction issued between two v_mfma_f32_32x32x16_bf16 of 32 cycles each):
 *     up to 4 vector-ALU instructions      ~0      (v_cvt_pk_f32_fp8 counts as two)
 *     ds_read_b128                         ~7      (16 alone: 1 KB at 64 B per clock and SIMD)
 *     ds_write_b128                        ~46     (1 KB at about 20 B per clock and SIMD; not hidden by anything)
 *     buffer_load_dwordx4 to registers     64 per KB and SIMD once the compute unit's 64 B per clock are in use, and
 *                                          four times that when every lane reads its own row (as an operand layout
 *                                          would need)
 *     buffer_load_dwordx4 ... lds          the same 64 B per clock, no register or LDS-store cost
 * So nothing is stored to LDS by a wave:
 *   - activations go from global memory to LDS by the load-to-LDS path, 32 NB tokens x 64 k per tile, whole 128-byte
 *     row segments per 8 lanes, four stages deep;
 *   - decoded weights never touch LDS: wave w owns rows 32 w .. 32 w + 31 of the workgroup's 128 and all its tokens,
 *     its lane (row i, half kg) takes 16 of the 32 code bytes of a quarter super-block of its row and decodes them
 *     straight into the matrix instruction's first-operand layout (8 consecutive k of one row per lane): no decode
 *     is done twice in the workgroup, and there is nothing to exchange. The raw blocks of a wave's rows come the same
 *     way as the activations (whole 144-byte blocks, consecutive lanes consecutive bytes; a lane reading its own
 *     row from global memory costs the memory pipe four times as much) and are read back by the wave itself;
 *   - per matrix instruction one ds_read_b128 (a 32-token x 16-k activation fragment) and about three vector
 *     instructions of decode.
 *
 * The formats differ in what a lane takes from its row's block (Q4_K: 16 code bytes per quarter; Q5_K: those
 * and 16 bytes of fifth bits per super-block; Q6_K: two runs of 16 nibble bytes and 16 bytes of bit pairs per half
 * super-block; Q8_0: the 32 codes of one block per tile, scales straight from memory) and in the arithmetic of a
 * piece; the tile loop is one template over a format description.
 *
 * k inside a tile is permuted so that a lane's 16 code bytes serve its four k-steps (Q4_K; the others alike): k-step s of lane half kg covers
 * the low (s < 2) or high nibbles of code bytes 16 kg + 8 (s & 1) .. + 7, i.e. tile k 32 (s >> 1) + 16 kg + 8 (s & 1) ..;
 * the activation fragment of that lane half is chunk 4 (s >> 1) + 2 kg + (s & 1) of the token's 128-byte row segment.
 *
 * LDS: four stages of [32 NB tokens][64 k] bf16 = 4 NB KB; 16-byte chunk c of token row r sits at chunk position
 * c ^ f(r), f = bits 1 and 2 of (r >> 1) & 7 swapped, so that the 16 rows of a fragment fetch hit 16 different
 * 16-byte bank groups. One tile = 4 NB slots of [matrix instruction, fragment fetch for the next k-step, side work],
 * nothing moves between slots; side work = the load-to-LDS requests of the tile three ahead and of the raw blocks
 * two super-blocks ahead, and the decode of the next tile in 44 to 88 pieces of at most two vector instructions. Before the last
 * k-step: wait for this wave's requests of the next tile, barrier (the next tile is complete; nobody reads the
 * stage that is requested next, its last fragments were fetched a k-step earlier).
 *
 * Fewer token blocks: a tile's decode costs the same whatever its tokens (9.0 vector instructions per matrix instruction, itself
 * included, at three blocks, 6.0 at five, 4.0 at eight, Q4_K), so that eight blocks cost least per token - a tile of 64 k in a full round of 256 workgroups takes 0.46 us
 * with four, 0.53, 0.61 and 0.78 with five, six and eight - and fewer win where eight would be padding or leave a second round of the chip
 * nearly empty. Three blocks fit a compute unit twice (at most 80 KB of LDS, 256 registers): 448 workgroups run at once, two waves
 * per SIMD. What bounds fewer blocks is the vector ALU, and start and drain: the matrix pipe is busy 28 and 37 % of a kernel of three blocks
 * (Q6_K, Q4_K), 26 and 32 of five. Against the better one of
 * 256 x 128 and 128 x 64 tiles, us (choose_token_blocks picks): Q4_K x 4096, 77 tokens 28672 rows 37.4 -> 31.8 (three), 128 tokens 41.3 -> 38.3
 * (four), 180 tokens 55 -> 48.6 (six), 300 tokens 12288 rows 51 -> 37.9 (five), 512 tokens 6144 rows 36.6 -> 32.9 (four). Q6_K 48.6 ->
 * 42.8, 53.5 -> 48.1, 65 -> 60.4, 57 -> 46.6, 46.6 -> 41.7. 128 x 128 tiles on eight waves, four row groups x two halves of K, were built and
 * are slower than four blocks here: 36.7 for 6144 rows at 512 tokens, a third of the waves' time at the barriers.
 *
 * Every wave keeps two sums per result, of k-steps 0 and 1 of the tiles and of 2 and 3, and adds them at the end: the 128 x 64 kernel's
 * two halves of K. So all tile shapes give the same bits, and which one a launch takes is free - the one that suits its tensors together.
 * (Where K is divided over workgroups the shape is a tensor's own choice, and one sum is kept: the second costs a launch 1 us. A
 * tensor that shares such a launch with its K whole keeps two.)
 */
#ifndef QLIN_GEMM_KQ_WAVE4_H
#define QLIN_GEMM_KQ_WAVE4_H
#include <utility>

#include "gemm_kq_formats.h"
#include "qlin_internal.h"

namespace qlin {

using namespace kq;

namespace {

constexpr int kBN = 128;

/* The four stages, 32 NB tokens x 64 k each, are separate objects: a fetch from one stage then never has to wait for a request into
 * another */
template <int NB, int ST> QLIN_INL uint8_t *stage_ptr() {
    __shared__ __attribute__((aligned(1024))) uint8_t w4_stage[NB * 4096];
    return w4_stage;
}

/* everything a slot touches; every member ends up in registers (all indices are constants after inlining) */
template <class Fmt, int NBLOCKS, int SUMS> struct Ctx {
    using F = Fmt;
    static constexpr int NB = NBLOCKS, S = 4 * NB, kSums = SUMS; /* token blocks; slots of a tile */
    floatx16 acc[SUMS][NB];  /* [SUMS 2: k-steps 0 and 1 of the tiles, 2 and 3][token block]: 32 rows x 32 tokens each */
    bf16x8 xf[2][NB];         /* activation fragments of the k-step in use and of the next: [k-step & 1][token block] */
    u32x4 wa[2][4];          /* decoded weights of the tile in use and of the next: [tile & 1][k-step] */
    u32x4 cur[F::kLaneVec + F::kExtraVec], nxt[F::kLaneVec + F::kExtraVec]; /* raw data of the super-block of the tile being
                                decoded, and of the next: kLaneVec vectors out of the LDS image, kExtraVec straight from memory */
    typename F::Scales sc;   /* of the super-block being decoded */
    Temps t;
    uint32_t xrd;            /* byte offset of this lane's fragment fetches in a stage: k-step 0, token block 0 */
    __amdgpu_buffer_rsrc_t w_rsrc, x_rsrc;
    uint32_t w_off[F::kReq], w_rd, w_swz, w_own, x_off[NB]; /* w_swz: see kSwizzle; w_own: byte offset of the lane's own
                                                               row in the weight tile */
    uint8_t *raw;            /* the workgroup's raw-block area in LDS */
    int wv, kg;              /* wave of the workgroup; lane half */
    int sb, n_sb;            /* super-block of the tile in use */
    float unit;
};


/* request Q (0 .. kReq - 1) of this wave for the raw blocks of super-block `sb` of its 32 rows (past the end of K: a
 * harmless re-read) */
template <int Q, class C> QLIN_INL void request_w(C &c, int sb) {
    dma16(c.w_rsrc, c.raw + (c.wv * C::F::kReq + Q) * 1024, c.w_off[Q], min(sb, c.n_sb - 1) * C::F::kBlockBytes);
}
/* vector J of this lane's raw data out of its row's image */
template <int J, class C> QLIN_INL u32x4 load_raw(C &c) {
    constexpr VecAt at = C::F::vec_at(J);
    return *reinterpret_cast<const u32x4 *>(c.raw + c.w_rd + ((uint32_t)(at.off + at.by_half * c.kg) ^ c.w_swz));
}

/* request I (below NB) of this wave for 64-k tile `tile` into stage ST: token rows 8 (NB wv + I) .. + 7, 128 bytes each */
template <int ST, int I, class C> QLIN_INL void request_x(C &c, int tile) {
    dma16(c.x_rsrc, stage_ptr<C::NB, ST>() + (C::NB * c.wv + I) * 1024, c.x_off[I], min(tile, 4 * c.n_sb - 1) * 128);
}

/* activation fragment of token block BJ, k-step S of stage ST */
template <int ST, int S, int BJ, class C> QLIN_INL bf16x8 load_frag(C &c) {
    return *reinterpret_cast<const bf16x8 *>(stage_ptr<C::NB, ST>() + (c.xrd ^ (uint32_t)C::F::frag_xor(S)) + BJ * 4096);
}

/* n items of side work over the first `slots` slots of a tile: those of slot T are first(T) .. first(T + 1) - 1 */
constexpr int first_of(int T, int n, int slots) { return T >= slots ? n : (T * n + slots - 1) / slots; }

/* slot T (0 .. 4 NB - 1) of tile 4 sb + U */
template <int U, int T, class C> QLIN_INL void slot(C &c) {
    using F = typename C::F;
    constexpr int NB = C::NB, S = C::S, s = T / NB, bj = T % NB;
    if constexpr (T == 3 * NB) {
        /* this wave's requests of the next tile have landed: younger are the NB of the tile after it, three quarters of those of the
         * one after that, the weight requests of a tile with U = 1 and the scale loads of one with U = 0 (all of them if
         * that was the tile before, those of its slots so far if it is this one) */
        constexpr int w_now = first_of(T, F::kReq, S), x_now = first_of(T, F::kExtraLoads, S);
        wait_vmcnt<NB + (3 * NB + 1) / 4 + (U == 0 ? x_now : 0) + (U == 1 ? w_now + F::kExtraLoads : 0) + (U == 2 ? F::kReq : 0)>();
        __builtin_amdgcn_s_barrier();
    }
    floatx16 &acc = c.acc[C::kSums == 2 ? s >> 1 : 0][bj];
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, c.wa[U & 1][s]), c.xf[s & 1][bj], acc, 0, 0, 0);
    c.xf[(s + 1) & 1][bj] = load_frag<(s == 3 ? (U + 1) & 3 : U), (s + 1) & 3, bj>(c);
    if constexpr (T % 4 == 2) request_x<(U + 3) & 3, T / 4>(c, 4 * c.sb + U + 3);
    /* U = 0: the raw data of the next super-block (requested three tiles ago) into registers; U = 1: request the
     * one after it into the same place; U = 3: the tile being decoded is the first of the next super-block, which
     * then becomes the one in work */
    auto some = [&](auto n, auto slots, auto fn) { /* (at most four per slot) */
        constexpr int N = decltype(n)::value, SL = decltype(slots)::value, i0 = first_of(T, N, SL), i1 = first_of(T + 1, N, SL);
        static_assert(i1 - i0 <= 4, "items of a slot");
        if constexpr (i0 < i1) fn(std::integral_constant<int, i0>{});
        if constexpr (i0 + 1 < i1) fn(std::integral_constant<int, i0 + 1>{});
        if constexpr (i0 + 2 < i1) fn(std::integral_constant<int, i0 + 2>{});
        if constexpr (i0 + 3 < i1) fn(std::integral_constant<int, i0 + 3>{});
    };
    using std::integral_constant;
    if constexpr (U == 0) {
        some(integral_constant<int, F::kLaneVec>{}, integral_constant<int, 3 * NB>{}, [&](auto i) { c.nxt[decltype(i)::value] = load_raw<decltype(i)::value>(c); });
        some(integral_constant<int, F::kExtraLoads>{}, integral_constant<int, S>{}, [&](auto i) { F::template extra_load<decltype(i)::value>(c, c.nxt, min(c.sb + 1, c.n_sb - 1)); });
    }
    if constexpr (U == 1) some(integral_constant<int, F::kReq>{}, integral_constant<int, S>{}, [&](auto i) { request_w<decltype(i)::value>(c, c.sb + 2); });
    if constexpr (U == 3) some(integral_constant<int, F::kLaneVec + F::kExtraVec>{}, integral_constant<int, S>{}, [&](auto i) { c.cur[decltype(i)::value] = c.nxt[decltype(i)::value]; });
    constexpr int n_pieces = F::kTilePieces + (U == 3 ? F::kPrepPieces : 0);
    constexpr int p0 = first_of(T, n_pieces, S), p1 = first_of(T + 1, n_pieces, S);
    /* (beside eight blocks there are fewer than two per slot, and a word's own order is as good) */
    constexpr auto nth = [](int p) constexpr { return NB == 8 ? p : tile_piece_at<F>(p); };
    auto piece = [&](auto pc) {
        constexpr int p = decltype(pc)::value;
        if constexpr (p < p1) {
            if constexpr (U == 3) {
                if constexpr (p < F::kPrepPieces) F::template prep<p>(c, c.nxt);
                else F::template tile_piece<0, 0, nth(p - F::kPrepPieces)>(c, c.nxt);
            } else {
                F::template tile_piece<U + 1, (U + 1) & 1, nth(p)>(c, c.cur);
            }
        }
    };
    piece(integral_constant<int, p0>{});
    piece(integral_constant<int, p0 + 1>{});
    piece(integral_constant<int, p0 + 2>{});
    piece(integral_constant<int, p0 + 3>{});
    piece(integral_constant<int, p0 + 4>{});
    piece(integral_constant<int, p0 + 5>{});
    piece(integral_constant<int, p0 + 6>{});
    piece(integral_constant<int, p0 + 7>{});
    static_assert(p1 - p0 <= 8, "at most eight pieces per slot");
    __builtin_amdgcn_sched_barrier(0);
}

template <int U, class C, int... T> QLIN_INL void run_tile(C &c, std::integer_sequence<int, T...>) { (slot<U, T>(c), ...); }
template <class C, int... P> QLIN_INL void prep_first(C &c, std::integer_sequence<int, P...>) { (C::F::template prep<P>(c, c.cur), ...); }
template <class C, int... P> QLIN_INL void decode_first(C &c, std::integer_sequence<int, P...>) { (C::F::template tile_piece<0, 0, P>(c, c.cur), ...); }
template <int ST, class C, int... I> QLIN_INL void request_tile(C &c, int tile, std::integer_sequence<int, I...>) { (request_x<ST, I>(c, tile), ...); }
template <class C, int... Q> QLIN_INL void request_raw(C &c, int sb, std::integer_sequence<int, Q...>) { (request_w<Q>(c, sb), ...); }
template <class C, int... J> QLIN_INL void load_cur(C &c, std::integer_sequence<int, J...>) { ((c.cur[J] = load_raw<J>(c)), ...); }
template <class C, int... J> QLIN_INL void load_cur_extra(C &c, std::integer_sequence<int, J...>) { (C::F::template extra_load<J>(c, c.cur, 0), ...); }
template <class C, int... B> QLIN_INL void load_first(C &c, std::integer_sequence<int, B...>) { ((c.xf[0][B] = load_frag<0, 0, B>(c)), ...); }

/* raw blocks of one super-block of each wave's 32 weight rows (32 x kPieces pieces, rounded up to whole requests) */
template <class F> QLIN_INL uint8_t *raw_ptr() {
    __shared__ __attribute__((aligned(1024))) uint8_t w4_raw[4 * F::kReq * 1024];
    return w4_raw;
}

/* one tile: this workgroup's super-blocks (`part`, of rows of n_sb_all) of token tile tile_m, in SUMS sums per result; `tid` = threadIdx.x */
template <class F, int NB, int SUMS> QLIN_INL void run_part(const KPart &part, const uint16_t *X, int n_sb_all, int n_tok, int ldx, int tile_m, int tid) {
    const int lane = tid & 63;
    const int n_sb = part.n_sb, n_rows = part.n_rows, ldy = part.ld, tile_n = part.tile;
    const uint8_t *W = part.W + (size_t)part.sb0 * F::kBlockBytes;
    float *Y = part.out;
    X += part.sb0 * 256;

    Ctx<F, NB, SUMS> c;
    constexpr int kBM = 32 * NB;
    c.raw = raw_ptr<F>();
    c.wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    c.n_sb = n_sb;
    c.unit = 1.0f / fp8_pair_lo(1u).x;
    const uint32_t row_bytes = (uint32_t)n_sb_all * F::kBlockBytes;
    /* Global loads are buffer loads: a descriptor of this workgroup's weight rows / token rows in scalar
     * registers, a 32-bit offset per lane that never changes, and a scalar offset that moves along K.
     * Weight role: lane (i = lane % 32, kg = lane / 32) owns row 32 wv + i; rows past the end re-read the last one
     * (decoded, never stored). Request q of a wave fills pieces 64 q .. 64 q + 63 of its 32 x kPieces. */
    const int li = lane & 31, kg = lane >> 5;
    const int w_rows = min(kBN, n_rows - tile_n * kBN);
    c.w_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(W) + (size_t)tile_n * kBN * row_bytes, 0,
                                                 (w_rows - 1) * row_bytes + (uint32_t)n_sb * F::kBlockBytes, 0x00020000);
    c.kg = kg;
#pragma unroll
    for (int q = 0; q < F::kReq; q++) {
        const int id = min(64 * q + lane, 32 * F::kPieces - 1); /* past the last piece: padding */
        const int part = F::kSwizzle ? (id % F::kPieces) ^ ((id / F::kPieces) & 15) : id % F::kPieces;
        c.w_off[q] = (uint32_t)min(32 * c.wv + id / F::kPieces, w_rows - 1) * row_bytes + F::piece_src(part);
    }
    c.w_rd = (uint32_t)(c.wv * F::kReq * 1024 + li * F::kPieces * 16);
    c.w_swz = F::kSwizzle ? (uint32_t)(li & 15) << 4 : 0u;
    c.w_own = (uint32_t)min(32 * c.wv + li, w_rows - 1) * row_bytes;
    /* Activation requests: request I of this wave fills 1 KB of a stage, lane l the 16 bytes at chunk position l % 8 of
     * token row 8 (NB wv + I) + l / 8, i.e. chunk (l % 8) ^ f(row) of that token's 128 bytes; tokens past the end
     * re-read the last one (never stored) */
    const int x_rows = min(kBM, n_tok - tile_m * kBM);
    c.x_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(X) + (size_t)tile_m * kBM * ldx, 0,
                                                 ((x_rows - 1) * ldx + n_sb * 256) * 2, 0x00020000);
#pragma unroll
    for (int i = 0; i < NB; i++) {
        const int row = 8 * (NB * c.wv + i) + (lane >> 3);
        c.x_off[i] = (uint32_t)min(row, x_rows - 1) * (uint32_t)(2 * ldx) + (uint32_t)((((lane & 7) ^ fsw(row))) << 4);
    }
    /* fragment fetches: token li of each block of 32; chunk 4 (s >> 1) + 2 kg + (s & 1) for the K-quants */
    c.xrd = (uint32_t)(li * 128 + (((F::kKgChunk * kg) ^ fsw(li)) << 4));

#pragma unroll
    for (int i = 0; i < NB; i++)
#pragma unroll
        for (int v = 0; v < 16; v++) {
            c.acc[0][i][v] = 0.0f;
            if constexpr (SUMS == 2) c.acc[1][i][v] = 0.0f;
        }

    /* ---- prologue: raw blocks of super-block 0 fetched and read back, those of super-block 1 and tiles 0..2
     * requested; tile 0 decoded; fragments of its k-step 0 fetched */
    c.sb = 0;
    load_cur_extra(c, std::make_integer_sequence<int, F::kExtraLoads>{});
    request_raw(c, 0, std::make_integer_sequence<int, F::kReq>{});
    request_tile<0>(c, 0, std::make_integer_sequence<int, NB>{});
    wait_vmcnt<NB>();
    load_cur(c, std::make_integer_sequence<int, F::kLaneVec>{});
    __builtin_amdgcn_s_waitcnt(0xC07F); /* lgkmcnt(0): the registers hold super-block 0 before its place is requested again */
    request_raw(c, 1, std::make_integer_sequence<int, F::kReq>{});
    request_tile<1>(c, 1, std::make_integer_sequence<int, NB>{});
    request_tile<2>(c, 2, std::make_integer_sequence<int, NB>{});
    prep_first(c, std::make_integer_sequence<int, F::kPrepPieces>{});
    decode_first(c, std::make_integer_sequence<int, F::kTilePieces>{});
    wait_vmcnt<2 * NB>(); /* tile 0 and the raw blocks of super-block 1 are in LDS as far as this wave's requests go */
    __builtin_amdgcn_s_barrier();
    load_first(c, std::make_integer_sequence<int, NB>{});

#pragma unroll 1
    for (int sb = 0; sb < n_sb; sb++) { /* one super-block of K = four tiles per pass */
        c.sb = sb;
        run_tile<0>(c, std::make_integer_sequence<int, 4 * NB>{});
        run_tile<1>(c, std::make_integer_sequence<int, 4 * NB>{});
        run_tile<2>(c, std::make_integer_sequence<int, 4 * NB>{});
        run_tile<3>(c, std::make_integer_sequence<int, 4 * NB>{});
    }
    wait_vmcnt<0>(); /* requests past the end of K are still on their way into LDS */

    /* C layout of the 32x32 MFMA: register v of lane l holds row 8 (v / 4) + 4 (l / 32) + v % 4 (a weight row), column
     * l % 32 (a token): four runs of four consecutive floats of one token's output row per lane */
#pragma unroll
    for (int bj = 0; bj < NB; bj++) {
        const int m = tile_m * kBM + 32 * bj + li;
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const int n = tile_n * kBN + 32 * c.wv + 8 * g + 4 * kg;
            if (m >= n_tok) continue;
            float *y = Y + (size_t)m * ldy + n;
            floatx4 a;
#pragma unroll
            for (int v = 0; v < 4; v++) {
                a[v] = c.acc[0][bj][4 * g + v];
                if constexpr (SUMS == 2) a[v] += c.acc[1][bj][4 * g + v];
            }
            store4(y, a, n_rows - n);
        }
    }
}

}  // namespace

template <class F, int NB, bool DIVIDED>
__global__ void __launch_bounds__(256)
gemm_kq_bf16_wave4_kernel(TileSet set, const uint16_t *__restrict__ X, int n_sb_all, int n_tok, int ldx, int m_tiles,
                          const KItems<DIVIDED> split) {
    /* consecutive workgroup ids land on different XCDs (id % 8), each with its own L2; the token tiles
     * that share one weight tile get ids 8 apart and meet in the same L2 */
    const int xcd = blockIdx.x & 7, slot_id = blockIdx.x >> 3;
    const int tile_m = slot_id % m_tiles;
    const int item = (slot_id / m_tiles) * 8 + xcd;
    if (item >= set.end2) return;
    /* this workgroup's super-blocks, and where its sums go */
    const KPart part = k_part(set, split, item, n_sb_all, n_tok);
    int tid = threadIdx.x;
    if constexpr (DIVIDED) {
        /* One branch per workgroup: a tensor that keeps its K whole beside divided ones has two sums here as well, as in a call of its own.
         * That costs such a launch 1 % (Q5_K 13568 + 3392 + 3392 rows x 13568 at 1009 tokens 563 -> 571 us), a launch for each kind 3.5 % in
         * the mean and up to 13 (Q5_K 10240 + 1100 + 1100 x 10240 at 899 282 -> 297, IQ4_NL 12032 + 1705 + 1705 x 12032 at 737 333 -> 379);
         * launches with divided tensors only take what they did. (The lane's number is opaque to the compiler in one branch, which
         * else computes both branches' offsets ahead of them and spills some.) */
        if (part.divided) run_part<F, NB, 1>(part, X, n_sb_all, n_tok, ldx, tile_m, tid);
        else {
            asm volatile("" : "+v"(tid));
            run_part<F, NB, 2>(part, X, n_sb_all, n_tok, ldx, tile_m, tid);
        }
    } else run_part<F, NB, 2>(part, X, n_sb_all, n_tok, ldx, tile_m, tid);
}

namespace {
template <class F, int NB>
hipError_t launch_wave4_blocks(const Wave4Call &c) {
    const int n_sb = c.n_cols / 256;
    const int m_tiles = (c.n_tok + 32 * NB - 1) / (32 * NB);
    TileSet set;
    const int n_tiles = fill_tile_set(set, c.n_mat, c.W, c.Y, c.n_rows, c.ldy, kBN, c.split);
    /* ids are dealt to 8 XCDs; pad the n-tile count to a multiple of 8 (surplus groups exit) */
    const int n_tiles_pad = (n_tiles + 7) / 8 * 8;
    const dim3 grid(n_tiles_pad * m_tiles), block(256);
    if (c.split.divides()) {
        if constexpr (NB == kLargeBlocks) {
            hipLaunchKernelGGL((gemm_kq_bf16_wave4_kernel<F, NB, true>), grid, block, 0, c.stream, set, c.X, n_sb, c.n_tok, c.ldx, m_tiles, k_items(c.split));
            launch_k_join(c.split, c.n_mat, c.Y, c.n_rows, c.n_tok, c.ldy, c.stream);
        } else return hipErrorInvalidValue;
    } else {
        hipLaunchKernelGGL((gemm_kq_bf16_wave4_kernel<F, NB, false>), grid, block, 0, c.stream, set, c.X, n_sb, c.n_tok, c.ldx, m_tiles, KItems<false>());
    }
    return hipGetLastError();
}
template <class F> hipError_t wave4_format(const Wave4Call &c) {
    switch (c.blocks) {
    case 3: return launch_wave4_blocks<F, 3>(c);
    case 4: return launch_wave4_blocks<F, 4>(c);
    case 5: return launch_wave4_blocks<F, 5>(c);
    case 6: return launch_wave4_blocks<F, 6>(c);
    case kLargeBlocks: return launch_wave4_blocks<F, kLargeBlocks>(c);
    default: return hipErrorInvalidValue;
    }
}
}  // namespace

}  // namespace qlin
#endif
