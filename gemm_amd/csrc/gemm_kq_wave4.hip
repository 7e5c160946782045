/*
 * gemm_kq_wave4.hip - the fused block-format x bf16 prefill GEMM (Q2_K ... Q6_K, Q8_0, IQ4_NL, IQ4_XS, Q4_0: the formats of
 * gemm_kq_formats.h) in tiles of 128 rows x 256 tokens, or 192, 160, 128, 96: four waves per workgroup, one per SIMD.
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
 * Fewer token blocks: a tile's decode costs the same whatever its tokens, about as much vector time as six blocks' matrix
 * instructions (Q4_K, one tile of 64 k on a chip of 224 workgroups: 0.41 us + 0.10 per block), so that eight blocks cost least per
 * token, and fewer win where eight would be padding or leave a second round of the chip nearly empty. Against the better one of
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
#include <climits>
#include <utility>

#include "gemm_kq_formats.h"
#include "qlin_internal.h"

#include <algorithm>
#include <climits>

namespace qlin {

using namespace kq;

namespace {

constexpr int kBN = 128, kLargeBlocks = 8;

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

/* adds the parts of K in order; a thread has R rows of a token, blockIdx.z is the tensor */
struct JoinOne { const float *buf; float *Y; int parts, n_rows, ldy; };
struct JoinSet { JoinOne a, b, c; };
template <int R>
__global__ void __launch_bounds__(256)
k_join_kernel(const JoinSet set, int n_tok) {
    typedef float vec __attribute__((ext_vector_type(R)));
    const int row = (blockIdx.x * 256 + threadIdx.x) * R, t = blockIdx.y;
    JoinOne j = set.a;
    if (blockIdx.z == 1) j = set.b;
    if (blockIdx.z == 2) j = set.c;
    if (row >= j.n_rows) return;
    const float *at = j.buf + (size_t)t * j.n_rows + row;
    vec sum = *reinterpret_cast<const vec *>(at);
#pragma unroll 4
    for (int p = 1; p < j.parts; p++) sum += *reinterpret_cast<const vec *>(at + (size_t)p * n_tok * j.n_rows);
    *reinterpret_cast<vec *>(j.Y + (size_t)t * j.ldy + row) = sum;
}

}  // namespace

void launch_k_join(const KSplit &split, int n_mat, float *const *Y, const int *n_rows, int n_tok, const int *ldy, hipStream_t stream) {
    JoinSet set = {};
    int n = 0, most = 0;
    bool wide = true; /* (a tensor's place in the workspace is 256-byte aligned) */
    for (int i = 0; i < n_mat; i++) {
        if (split.parts[i] < 2) continue;
        (n == 0 ? set.a : n == 1 ? set.b : set.c) = {split.buf[i], Y[i], split.parts[i], n_rows[i], ldy[i]};
        wide = wide && n_rows[i] % 4 == 0 && ldy[i] % 4 == 0 && ((uintptr_t)Y[i] & 15) == 0;
        most = std::max(most, n_rows[i]);
        n++;
    }
    const int per = 256 * (wide ? 4 : 1);
    hipLaunchKernelGGL(wide ? k_join_kernel<4> : k_join_kernel<1>, dim3((most + per - 1) / per, n_tok, n), dim3(256), 0, stream, set, n_tok);
}

namespace {
template <class F, int NB>
hipError_t launch_wave4_blocks(int n_mat, const void *const *W, const uint16_t *X, float *const *Y, const int *n_rows, int n_cols,
                        int n_tok, int ldx, const int *ldy, KSplit split, hipStream_t stream) {
    const int n_sb = n_cols / 256;
    const int m_tiles = (n_tok + 32 * NB - 1) / (32 * NB);
    TileSet set;
    const int n_tiles = fill_tile_set(set, n_mat, W, Y, n_rows, ldy, kBN, split);
    /* ids are dealt to 8 XCDs; pad the n-tile count to a multiple of 8 (surplus groups exit) */
    const int n_tiles_pad = (n_tiles + 7) / 8 * 8;
    const dim3 grid(n_tiles_pad * m_tiles), block(256);
    if (split.divides()) {
        if constexpr (NB == kLargeBlocks) {
            hipLaunchKernelGGL((gemm_kq_bf16_wave4_kernel<F, NB, true>), grid, block, 0, stream, set, X, n_sb, n_tok, ldx, m_tiles, k_items(split));
            launch_k_join(split, n_mat, Y, n_rows, n_tok, ldy, stream);
        } else return hipErrorInvalidValue;
    } else {
        hipLaunchKernelGGL((gemm_kq_bf16_wave4_kernel<F, NB, false>), grid, block, 0, stream, set, X, n_sb, n_tok, ldx, m_tiles, KItems<false>());
    }
    return hipGetLastError();
}
template <class F>
hipError_t launch_wave4(int blocks, int n_mat, const void *const *W, const uint16_t *X, float *const *Y, const int *n_rows, int n_cols,
                        int n_tok, int ldx, const int *ldy, KSplit split, hipStream_t stream) {
    switch (blocks) {
    case 3: return launch_wave4_blocks<F, 3>(n_mat, W, X, Y, n_rows, n_cols, n_tok, ldx, ldy, split, stream);
    case 4: return launch_wave4_blocks<F, 4>(n_mat, W, X, Y, n_rows, n_cols, n_tok, ldx, ldy, split, stream);
    case 5: return launch_wave4_blocks<F, 5>(n_mat, W, X, Y, n_rows, n_cols, n_tok, ldx, ldy, split, stream);
    case 6: return launch_wave4_blocks<F, 6>(n_mat, W, X, Y, n_rows, n_cols, n_tok, ldx, ldy, split, stream);
    case kLargeBlocks: return launch_wave4_blocks<F, kLargeBlocks>(n_mat, W, X, Y, n_rows, n_cols, n_tok, ldx, ldy, split, stream);
    default: return hipErrorInvalidValue;
    }
}
}  // namespace

bool gemm_kq_wave4_covers(uint32_t type) {
    return type == T_Q4_K || type == T_Q5_K || type == T_Q6_K || type == T_Q8_0 || type == T_IQ4_NL || type == T_IQ4_XS ||
           type == T_Q4_0 || type == T_Q2_K || type == T_Q3_K;
}

/* Estimates, in us, for the tensors of a launch in each shape of tile. A super-block costs a full round of 256 workgroups what the
 * table says (the 128 x 64 kernel's: up to 256 workgroups, and 512), a round that leaves compute units idle less - the clock is higher
 * then, the more so the more blocks; three blocks fit a compute unit's LDS twice. Row tiles are dealt to 8 XCDs of 32 compute units.
 * The results go to memory at 3.3 TB/s beside that. Fitted to 3700 measured products of nine formats (640 to 28672 rows x 1024 to
 * 14336 columns, 77 to 4096 tokens, runs long enough that the power limit counts); an estimate errs by 3.8 % in the mean. */
static constexpr int kTokenBlocks[6] = {0, 3, 4, 5, 6, kLargeBlocks};
static void tile_us(uint32_t type, int n_mat, const int *n_rows, int n_cols, int n_tok, double us[6]) {
    struct Cost { float small_256, small_512, b[5]; };
    Cost c;
    switch (type) {
    case T_Q4_K: c = {1.18f, 2.07f, {1.45f, 1.83f, 2.10f, 2.44f, 3.10f}}; break;
    case T_Q5_K: c = {1.25f, 2.20f, {1.61f, 2.02f, 2.28f, 2.67f, 3.20f}}; break;
    case T_Q6_K: c = {1.55f, 2.69f, {2.01f, 2.37f, 2.70f, 3.09f, 3.61f}}; break;
    case T_Q8_0: c = {2.03f, 3.52f, {2.42f, 2.83f, 3.07f, 3.44f, 3.95f}}; break;
    case T_IQ4_NL: c = {1.36f, 2.30f, {1.83f, 2.18f, 2.40f, 2.82f, 3.33f}}; break;
    case T_IQ4_XS: c = {1.46f, 2.33f, {1.85f, 2.22f, 2.47f, 2.89f, 3.42f}}; break;
    case T_Q4_0: c = {1.18f, 2.09f, {1.47f, 1.86f, 2.13f, 2.51f, 3.10f}}; break;
    case T_Q2_K: c = {1.13f, 1.96f, {1.37f, 1.74f, 2.05f, 2.35f, 3.05f}}; break;
    default: c = {1.28f, 2.21f, {1.59f, 1.93f, 2.21f, 2.59f, 3.18f}}; break; /* Q3_K */
    }
    constexpr float kIdle[5] = {0.97f, 0.90f, 0.865f, 0.85f, 0.825f}; /* of a round's time, where at most 112 workgroups run */
    long long rows = 0, rows128 = 0, rows64 = 0;
    for (int i = 0; i < n_mat; i++) {
        rows += n_rows[i];
        rows128 += ((long long)n_rows[i] + 127) / 128;
        rows64 += ((long long)n_rows[i] + 63) / 64;
    }
    const auto workgroups = [&](long long row_tiles, int tokens) { return (row_tiles + 7) / 8 * 8 * ((n_tok + tokens - 1) / tokens); };
    const double fixed = 3.3 + 1.2e-6 * rows * n_tok;
    const long long n_small = workgroups(rows64, 128), rest_small = n_small % 512;
    double rounds = (double)(n_small / 512) * c.small_512;
    if (rest_small > 256) rounds += c.small_256 + (c.small_512 - c.small_256) * (0.64 + 0.36 * (rest_small - 256) / 256);
    else if (rest_small > 0) rounds += c.small_256 * (0.73 + 0.27 * rest_small / 507.0);
    us[0] = fixed + n_cols / 256 * rounds;
    for (int i = 0; i < 5; i++) {
        const int nb = kTokenBlocks[i + 1];
        const long long n = workgroups(rows128, 32 * nb), per = nb == 3 ? 512 : 256, rest = n % per;
        rounds = (double)(n / per) * (nb == 3 ? 1.98 : 1.0);
        if (rest > 256) rounds += 1.0 + 0.98 * (0.6 + 0.4 * (rest - 256) / 256);
        else if (rest > 0) {
            const double x = std::min(1.0, std::max(0.0, (rest - 112) / 112.0));
            rounds += kIdle[i] + (1 - kIdle[i]) * x * x * x;
        }
        us[i + 1] = fixed + n_cols / 256 * c.b[i] * rounds;
    }
}

/* Which kernel takes a prefill GEMM of a format with a fused kernel, beyond the token counts of the few-token kernels.
 * 200 or more 256-token x 128-row tiles fill the chip: the large-tile kernel - up to a token count, because it decodes
 * the weights again every 256 tokens, which costs more the more there is to decode, while decoding once into a workspace
 * costs 27 - 38 us whatever the token count (14336 x 4096, large tiles against decode + the vendor library's product, us:
 * at 512 tokens Q4_K 61 / 86, Q5_K 62 / 92, Q6_K 66 / 84, Q8_0 71 / 83, IQ4_NL 62 / 95, IQ4_XS 68 / 99, Q4_0 62 / 81,
 * Q2_K 59 / 82, Q3_K 62 / 91; at 1024 118 / 125, 121 / 135, 131 / 126, 139 / 121, 123 / 132, 133 / 139, 122 / 120,
 * 117 / 120, 127 / 128; at 1536 Q4_K 181 / 190, Q5_K 185 / 195, Q6_K 206 / 184, Q8_0 216 / 177; at 2048 267 / 244,
 * 262 / 260, 273 / 240, 311 / 224, 279 / 254, 305 / 270, 272 / 241, 251 / 222, 261 / 253).
 * Fewer large tiles: the small-tile kernel, up to a token count per format (small tiles / decode + library, us, at
 * 4096 x 4096 and 4096 x 14336 with 512 tokens, the same two with 1024, 6144 x 4096 with 768, 14336 x 4096 with 256:
 * Q4_K 24 / 43, 72 / 97, 42 / 52, 133 / 153, 57 / 59, 39 / 75; Q5_K 25 / 44, 74 / 104, 43 / 54, 139 / 158, 59 / 61, 41 / 80;
 * Q6_K 29 / 40, 85 / 96, 49 / 51, 163 / 154, 68 / 57, 47 / 71; Q8_0 35 / 38, 109 / 97, 64 / 49, 216 / 152, 91 / 55, 62 / 75;
 * IQ4_NL 27 / 45, 80 / 108, 46 / 55, 148 / 161, 63 / 63, 44 / 88; IQ4_XS 27 / 45, 82 / 110, 47 / 55, 154 / 162, 64 / 63,
 * 45 / 80; Q4_0 24 / 41, 72 / 91, 41 / 50, 133 / 144, 57 / 56, 39 / 72; Q2_K 24 / 42, 70 / 94, 41 / 52, 132 / 149, 55 / 58,
 * 38 / 74; Q3_K 26 / 45, 75 / 102, 44 / 54, 144 / 160, 61 / 61, 42 / 82).
 * Those lines are for tensors of any size; smaller ones, whose tiles end in fewer or fuller rounds, gain beyond them. There the
 * estimates decide (tile_us; decode + library: 10.7 us, the decode 0.53 us per million weights, the product 1.48 PFLOP/s and its
 * results). The library's errs by a tenth, so that 10 % are asked for, of Q8_0 14: at 7 % Q6_K 1024 x 3584 at 1139 tokens and at 10 %
 * Q8_0 2048 x 2048 at 863 lost 2 us. us, decode + library / tiles: Q6_K 2048 x 2048 at 640 tokens 23.7 / 15.8, 2560 x 6912 at 640
 * 48 / 39, 2048 x 4096 at 1024 36 / 28; Q8_0 11008 x 1024 at 328 29.5 / 21.2; IQ4_NL 2048 x 2048 at 1300 28 / 22; Q4_K 4096 x 14336 at
 * 2048 235 / 201; Q2_K 4096 x 5120 at 3904 134 / 158, left alone. Of 837 random products past the lines 110 take tiles, in 0.84 of the
 * time (one is slower by more than 3 %); their error against 64 bits is 0.7 of that of the library's product.
 * Without a workspace there is no decode + dense route to prefer.
 * Up to 128 tokens half of a large tile is empty: small tiles whatever their number (77 tokens 28672 x 4096 large / small: Q4_K
 * 51 / 38, Q5_K 52 / 41, Q6_K 57 / 48; 128 tokens 65536 x 1024 Q4_K 1.26 times, IQ4_XS 1.27, Q3_K 1.30; Q8_0 even). Past 128
 * tokens by how often the chip has to go round: 256 large tiles (their row tiles are padded to eights) run at a time, 512 small
 * ones, and a small round costs 0.82 of a large one, its last part less the less there is of it (time of small tiles over large,
 * Q4_K ... Q6_K at 4096 columns: one round of large tiles, 512 small ones 0.82 - 0.89, 576 to 768 1.08 - 1.24, 1000 1.24 - 1.37;
 * two rounds, 792 to 960 small ones 0.71 - 0.81, 1160 0.92 - 0.98, 1400 1.06 - 1.14, 1840 1.31 - 1.46; three, 1560 0.81 - 0.87,
 * 2080 1.04 - 1.13, 2800 1.27 - 1.42; Q8_0's small tiles cost 1.2 times as much).
 * Tensors share a launch only if each takes the same kernel by itself, so the rounds count for those that come with others only
 * where they hold for the company too. Half to twice as many rows as columns (a Q, whose K and V take small tiles): large tiles from
 * 200 on, as for tensors of any size before (Q4_K Q, K and V of 4096 + 1024 + 1024 rows x 4096 at 1280 tokens shared / Q apart in large
 * tiles 80 / 99, 5120 + 1024 + 1024 x 5120 at 1024 97 / 119). More, below eight times (gate and up): by rounds where one tensor and the
 * pair agree, else the same (2 x 10240 x 2560 Q2_K at 984 tokens large / small tiles 117 / 134, 2 x 5888 x 1536 Q4_K at 1440 76 / 81). */
static bool small_by_rounds(uint32_t type, long long n_rows, int n_tok, int n_mat) {
    const long long padded = ((n_rows + 127) / 128 * n_mat + 7) / 8 * 8 * ((n_tok + 255) / 256), rounds = (padded + 255) / 256;
    return (n_rows + 63) / 64 * n_mat * ((n_tok + 127) / 128) <= (rounds == 1 || type == T_Q8_0 ? 512 : 650) * rounds;
}
FusedTile choose_fused_tile(uint32_t type, int n_rows, int n_cols, int n_tok, int ldx, bool have_workspace) {
    if (!gemm_kq_wave4_covers(type) || n_cols % 256 != 0 || ldx >= (1 << 22)) return kFusedNone;
    const long long large_tiles = ((long long)n_rows + 127) / 128 * ((n_tok + 255) / 256);
    /* token counts up to which the large-tile and the small-tile kernel measured faster than decode + dense */
    int large_max = 512, small_max = 256; /* Q8_0 */
    switch (type) {
    case T_Q4_K: case T_Q5_K: large_max = 1536; small_max = INT_MAX; break;
    case T_Q4_0: case T_Q2_K: case T_Q3_K: large_max = 1024; small_max = INT_MAX; break;
    case T_IQ4_NL: large_max = 1536; small_max = 1024; break;
    case T_IQ4_XS: large_max = 1024; small_max = 1024; break;
    case T_Q6_K: small_max = 512; break;
    default: break;
    }
    bool large_ok = n_tok <= large_max || !have_workspace, small_ok = n_tok <= small_max || !have_workspace;
    /* beyond: the estimates, in the range they were measured over (256 rows x 2304 IQ4_NL at 1860 tokens would lose 2 us; Q8_0's K
     * and V of a model wider than 11008 divide K at such token counts, and would part from a Q in tiles) */
    if ((!large_ok || !small_ok) && n_rows >= 640 && n_cols <= (type == T_Q8_0 ? 11008 : 14336)) {
        double us[6];
        tile_us(type, 1, &n_rows, n_cols, n_tok, us);
        const double weights = (double)n_rows * n_cols, results = (double)n_rows * n_tok;
        if (*std::min_element(us, us + 6) < (type == T_Q8_0 ? 0.86 : 0.9) * (10.7 + 0.53e-6 * weights + 1.352e-9 * weights * n_tok + 1.41e-3 * n_cols + 0.773e-6 * results))
            large_ok = small_ok = true;
    }
    if (large_tiles >= 200 && !large_ok) return kFusedNone;
    if (n_tok > 128 && large_ok && small_ok) {
        bool small = small_by_rounds(type, n_rows, n_tok, 1);
        const bool q = n_rows > n_cols / 2 && n_rows <= 2LL * n_cols, gate = n_rows > 2LL * n_cols && n_rows < 8LL * n_cols;
        if (q || (gate && small != small_by_rounds(type, n_rows, n_tok, 2))) small = large_tiles < 200;
        return small ? kFusedSmall : kFusedLarge;
    }
    if (large_tiles >= 200 && (n_tok > 128 || type == T_Q8_0)) return kFusedLarge;
    return small_ok ? kFusedSmall : kFusedNone;
}

/* Long rows on few tiles: K divided over workgroups, the parts added by a second launch (k_join_kernel). A chip of 256 compute
 * units with 64 tiles of a 4096 x 14336 product works through 56 super-blocks four times slower than it could; the tile
 * kernels' parts read no activation and no weight twice, but their sums go through memory (8 bytes per part and result) and
 * the second launch costs 3.5 us. Measured, us, one piece (few-token kernel to 128 tokens, then tiles, or decode + library) / divided, Q4_K:
 * 4096 x 14336 with 77, 128, 160, 256, 384, 512, 768 tokens 31.8 / 26.4, 45 / 29.4, 67 / 39, 69 / 44, 71 / 63, 81 / 68, 121 / 97; 2560 x 6912
 * with 128, 160, 256 19.5 / 15.8, 28 / 18, 31 / 19.5; 2048 x 5632 18.6 / 14.2, 23.5 / 15.4, 25 / 17.3; Q6_K 4096 x 14336 with 256, 768 83 / 47, 133 /
 * 106. Not below 17 super-blocks: 4096 x 4096 gains nothing (160 tokens 18.9 / 17.9, 512 23.6 / 32).
 * The estimates, in us, are fitted to such figures; they err by a tenth, so that a gain of less than 13 % is left alone. Over 500
 * random products of 256 to 8192 rows x 5632 to 16384 columns that divide: 0.60 of the time in one piece in the geometric mean, two slower, by 3 %.
 * Not a tensor that may come with others (may_share) where their one launch, in one piece, costs less than a launch in parts
 * and its join, or than one of them apart: a tensor's results are the same in a call of several and in one of its own. us, Q4_K unless said,
 * undivided in one launch / divided and sharing what they can:
 *   128 tokens: 5120 + 1024 + 1024 rows x 5120, Q in the few-token kernel, K and V not, 28 / 47; three of 5376 x 5376 IQ4_NL at 94 34 / 42;
 *     but 8192 + 1024 + 1024 x 8192 at 77 68 / 42 (K and V alone are few-token products there), three of 8192 x 8192 at 77 69 / 69
 *   more tokens: 5120 + 1024 + 1024 x 5120 at 256 29 / 36, 4096 + 2048 + 2048 x 5376 at 256 32 / 41, 6144 + 1024 + 1024 x 6144 at 512 61 / 71;
 *     Q8_0 8192 + 512 + 512 x 8192 at 179, Q in large tiles then, 108 / 169
 * That leaves on the table 8192 x 8192 Q6_K alone at 512 97 / 81, 1024 x 5120 alone at 256 20.6 / 13. K and V of 1536 rows and more in models
 * 5632 wide and wider divide, since a down product of a small model has their shape (2048 x 5632 at 256 24.5 / 16.7): undivided
 * in one launch / a call each / now 8192 + 2048 + 2048 x 8192 at 256 73 / 86 / 69, at 512 118 / 138 / 123, 6144 + 1536 + 1536 x 6144 at 256 54 /
 * 64 / 46, at 354 56 / 86 / 63; Q5_K 6656 + 1664 + 1664 x 6656 at 268 60 / 89 / 70. */
static bool may_share(uint32_t type, int n_rows, int n_cols, int n_tok, int ldx, FusedTile tile) {
    if (n_tok <= 128) /* K and V beside a Q of n_cols rows in the few-token kernel; three tensors of this shape that the chip takes at once */
        return fewtok_takes(type, n_cols, n_cols, n_tok, ldx) || (n_rows > n_cols / 2 && 3 * (((long long)n_rows + 63) / 64) <= 256);
    if (n_rows > n_cols / 2) return true;  /* Q (and what has its shape), gate, up */
    if (n_cols < 22 * 256) return true;    /* K and V of a model 4352 to 5376 wide */
    if (n_rows >= 1536 && n_cols < 6LL * n_rows) return false;
    for (const long long q20 : {15, 20, 32}) /* K and V of few rows, where a Q of 0.75 to 1.6 times n_cols rows takes the same tiles */
        if (choose_fused_tile(type, (int)std::min(q20 * n_cols / 20, (long long)INT_MAX), n_cols, n_tok, ldx, true) == tile) return true;
    return false;
}
FusedSplit choose_fused_split(uint32_t type, int n_rows, int n_cols, int n_tok, int ldx, size_t workspace_bytes, FusedTile tile, bool few) {
    const int n_sb = n_cols / 256;
    if (!gemm_kq_wave4_covers(type) || n_cols % 256 != 0 || n_sb < 17 || ldx >= (1 << 22) || n_tok < 65 || n_tok > 1024 ||
        may_share(type, n_rows, n_cols, n_tok, ldx, tile))
        return {tile, 1};
    double small = 1.0, large = 1.0, fewf = 1.0; /* the formats' times against Q4_K's */
    switch (type) {
    case T_Q5_K: small = 1.03; large = 1.02; break;
    case T_Q6_K: small = 1.2; large = 1.1; fewf = 1.08; break;
    case T_Q8_0: small = 1.65; large = 1.2; fewf = 1.1; break;
    case T_IQ4_NL: small = 1.15; large = 1.03; break;
    case T_IQ4_XS: small = 1.13; large = 1.13; break;
    case T_Q3_K: small = 1.06; large = 1.03; break;
    default: break;
    }
    const double results = (double)n_rows * n_tok, weights = (double)n_rows * n_cols;
    const auto joined = [&](int parts) { return parts > 1 ? 3.5 + parts * results * 8.0 / 4e6 : 0.0; };
    const auto small_us = [&](int parts) {
        const long long items = ((long long)n_rows + 63) / 64 * ((n_tok + 127) / 128) * parts;
        const double rounds = parts > 1 ? (double)((items + 255) / 256) : std::max(1.0, items / 256.0);
        return 4.5 + (n_sb + parts - 1) / parts * rounds * small * (0.65 + 0.008 * n_sb + 0.3 * std::min(1.0, items / 256.0)) + joined(parts);
    };
    const auto large_us = [&](int parts) {
        const long long items = (((long long)n_rows + 127) / 128 * parts + 7) / 8 * 8 * ((n_tok + 255) / 256); /* dealt to 8 XCDs of 32 units: 84 x 3 are two rounds */
        return 9.0 + (n_sb + parts - 1) / parts * ((items + 255) / 256) * large * (2.1 + 0.7 * std::min(1.0, items / 224.0)) + joined(parts);
    };
    double one; /* in one piece */
    if (few) one = 4.0 + fewf * n_sb * (0.1 + 0.0048 * (n_tok <= 80 ? 80 : n_tok <= 96 ? 96 : 128)) * (0.7 + 0.3 * std::min(1.0, n_rows / 4096.0));
    else if (tile == kFusedSmall) one = small_us(1);
    else if (tile == kFusedLarge) one = large_us(1);
    else one = 5.0 + weights * 2.8 / 4.2e6 + 2.0 * weights * n_tok / (1.25e9 * (0.4 + 0.6 * std::min(1.0, results / 6e6)));
    FusedSplit best = {tile, 1};
    double best_us = 0.87 * one;
    for (int parts = 2; parts <= 16 && parts <= n_sb / 2 && parts * results * sizeof(float) <= (double)workspace_bytes; parts++) {
        if (const double t = small_us(parts); t < best_us) { best_us = t; best = {kFusedSmall, parts}; }
        if (const double t = large_us(parts); n_tok > 128 && t < best_us) { best_us = t; best = {kFusedLarge, parts}; }
    }
    return best;
}

hipError_t launch_fused_split(FusedSplit s, uint32_t type, const void *W, const uint16_t *X, float *Y, int n_rows, int n_cols, int n_tok,
                              int ldx, int ldy, void *workspace, hipStream_t stream) {
    KSplit split;
    split.buf[0] = (float *)workspace;
    split.parts[0] = s.parts;
    return s.tile == kFusedLarge ? launch_gemm_kq_bf16_wave4_multi(type, kLargeBlocks, 1, &W, X, &Y, &n_rows, n_cols, n_tok, ldx, &ldy, stream, split)
                                 : launch_gemm_kq_bf16_wave4s_multi(type, 1, &W, X, &Y, &n_rows, n_cols, n_tok, ldx, &ldy, stream, split);
}

/* How many token blocks the tiles of a launch have (0: the 128-token x 64-row kernel), of tensors that take `tile` each by itself: the
 * least of tile_us. All shapes give the same bits, so the tensors of a launch are looked at together. Over 198 products of nine formats
 * (2048 to 28672 rows x 2048 to 4096 and 14336 columns, 77 to 1024 tokens) the choice costs 0.3 % of the best kernel's time and takes
 * 0.94 of what `tile` does (one tensor). A gain of less than 4 % is left alone: at 2 % pairs of 5632 x 1536 IQ4_XS at
 * 557 tokens lost 1 %. */
int choose_token_blocks(uint32_t type, FusedTile tile, int n_mat, const int *n_rows, int n_cols, int n_tok) {
    double us[6];
    tile_us(type, n_mat, n_rows, n_cols, n_tok, us);
    int best = tile == kFusedLarge ? 5 : 0;
    double best_us = 0.96 * us[best];
    for (int i = 0; i < 6; i++)
        if (us[i] < best_us) { best = i; best_us = us[i]; }
    return kTokenBlocks[best];
}

hipError_t launch_fused_tiles(FusedTile tile, uint32_t type, int n_mat, const void *const *W, const uint16_t *X, float *const *Y, const int *n_rows,
                              int n_cols, int n_tok, int ldx, const int *ldy, hipStream_t stream) {
    if (tile == kFusedNone) return hipErrorInvalidValue;
    const int blocks = choose_token_blocks(type, tile, n_mat, n_rows, n_cols, n_tok);
    return blocks ? launch_gemm_kq_bf16_wave4_multi(type, blocks, n_mat, W, X, Y, n_rows, n_cols, n_tok, ldx, ldy, stream)
                  : launch_gemm_kq_bf16_wave4s_multi(type, n_mat, W, X, Y, n_rows, n_cols, n_tok, ldx, ldy, stream);
}

hipError_t launch_fused_tile(FusedTile tile, uint32_t type, const void *W, const uint16_t *X, float *Y, int n_rows,
                             int n_cols, int n_tok, int ldx, int ldy, hipStream_t stream) {
    return launch_fused_tiles(tile, type, 1, &W, X, &Y, &n_rows, n_cols, n_tok, ldx, &ldy, stream);
}

hipError_t launch_gemm_kq_bf16_wave4_multi(uint32_t type, int blocks, int n_mat, const void *const *W, const uint16_t *X,
                                           float *const *Y, const int *n_rows, int n_cols, int n_tok, int ldx,
                                           const int *ldy, hipStream_t stream, KSplit split) {
    if (n_mat < 1 || n_mat > 3) return hipErrorInvalidValue;
    switch (type) {
    case T_Q4_K: return launch_wave4<FQ4K>(blocks, n_mat, W, X, Y, n_rows, n_cols, n_tok, ldx, ldy, split, stream);
    case T_Q5_K: return launch_wave4<FQ5K>(blocks, n_mat, W, X, Y, n_rows, n_cols, n_tok, ldx, ldy, split, stream);
    case T_Q6_K: return launch_wave4<FQ6K>(blocks, n_mat, W, X, Y, n_rows, n_cols, n_tok, ldx, ldy, split, stream);
    case T_Q8_0: return launch_wave4<FQ8_0>(blocks, n_mat, W, X, Y, n_rows, n_cols, n_tok, ldx, ldy, split, stream);
    case T_IQ4_NL: return launch_wave4<FIQ4NL>(blocks, n_mat, W, X, Y, n_rows, n_cols, n_tok, ldx, ldy, split, stream);
    case T_IQ4_XS: return launch_wave4<FIQ4XS>(blocks, n_mat, W, X, Y, n_rows, n_cols, n_tok, ldx, ldy, split, stream);
    case T_Q4_0: return launch_wave4<FQ4_0>(blocks, n_mat, W, X, Y, n_rows, n_cols, n_tok, ldx, ldy, split, stream);
    case T_Q2_K: return launch_wave4<FQ2K>(blocks, n_mat, W, X, Y, n_rows, n_cols, n_tok, ldx, ldy, split, stream);
    case T_Q3_K: return launch_wave4<FQ3K>(blocks, n_mat, W, X, Y, n_rows, n_cols, n_tok, ldx, ldy, split, stream);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace qlin
