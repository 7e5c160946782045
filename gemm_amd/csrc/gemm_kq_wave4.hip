/*
 * gemm_kq_wave4.hip - which prefill products the tile kernels take (gemm_kq_wave4.h: 128 rows, gemm_kq_wave4s.hip: 64), in which tiles
 * and in how many parts of K; the launch by format, and the launch that adds the parts.
 */
#include "qlin_internal.h"

#include <algorithm>
#include <climits>

namespace qlin {

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

bool gemm_kq_wave4_covers(uint32_t type) {
    return type == T_Q4_K || type == T_Q5_K || type == T_Q6_K || type == T_Q8_0 || type == T_IQ4_NL || type == T_IQ4_XS ||
           type == T_Q4_0 || type == T_Q2_K || type == T_Q3_K;
}

/* Estimates, in us, for the tensors of a launch in each shape of tile. A super-block costs a full round of 256 workgroups what the
 * table says (the 128 x 64 kernel's: 256 workgroups beside more, and 512), a round that leaves compute units idle less - the clock is
 * higher then, the more so the more blocks; three blocks fit a compute unit's LDS twice. Row tiles are dealt to 8 XCDs of 32 compute units.
 * The results go to memory at 3.3 TB/s beside that. Fitted to 3700 measured products of nine formats (640 to 28672 rows x 1024 to
 * 14336 columns, 77 to 4096 tokens, few of them past 2048, runs long enough that the power limit counts), fractions of a round
 * included: 0.73 + 0.27 of 507ths of one (of up to 256 workgroups; of 256ths it would be 7 % off from 130 on). On another card and in short
 * runs, where the power limit does not count, 1250 products of that range err by 7 % in the mean.
 * The 128 x 64 kernel reads X twice as often for a result, and past 2048 tokens the 64 workgroups that an XCD runs at a time no longer
 * meet on the same tokens in its L2, four row tiles on each: measured over estimated without the factor 1.15 (up to 1.8) at 2049 to 2560
 * tokens, 1.4 to 3072, 1.55 to 4096, 1.6 from there to 16384; with 1024 to 1792 columns 1.09, 1.22, 1.5 and 1.5, with fewer 0.92 to 1.18.
 * Not of fewer than 640 rows: there it is 1.1 to 1.6, but the other shapes are as far off where it counts, and with the factor two tensors
 * of 188 rows x 6400 Q8_0 at 3359 tokens went to large tiles, 54 -> 77 us. Beyond what it was fitted to an estimate errs by more: rows of
 * 256 to 768 elements 0.75 to 1.05 of the time, 28676 to 160000 rows 0.91 to 0.99, past 4096 tokens 0.83 to 0.98, 14592 to 28672 columns
 * 0.97 to 1.15. */
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
    const double past = n_cols < 1024 || rows < 640 ? 0.0 : std::min(1.0, std::max(0.0, (n_tok - (n_cols < 2048 ? 2304 : 2048)) / 1280.0));
    us[0] = (fixed + n_cols / 256 * rounds) * (1.0 + 0.6 * past);
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

/* What takes a prefill GEMM of a format with a fused kernel, beyond the token counts of the few-token kernels: decode + library, given a
 * workspace, or tiles, and of those the class, large or small. A class is no kernel any more: every shape of tile gives the same bits,
 * and choose_token_blocks picks one for the tensors of a launch. It says which tensors may share a launch (those of one class by themselves),
 * which kernel divides K, and which shape stays where no other is estimated to gain enough. The figures below are of 256-token x 128-row
 * (large) and 128-token x 64-row tiles (small).
 * 200 or more large tiles fill the chip: the large class - up to a token count, because it decodes
 * the weights again every 256 tokens, which costs more the more there is to decode, while decoding once into a workspace
 * costs 27 - 38 us whatever the token count (14336 x 4096, large tiles against decode + the vendor library's product, us:
 * at 512 tokens Q4_K 61 / 86, Q5_K 62 / 92, Q6_K 66 / 84, Q8_0 71 / 83, IQ4_NL 62 / 95, IQ4_XS 68 / 99, Q4_0 62 / 81,
 * Q2_K 59 / 82, Q3_K 62 / 91; at 1024 118 / 125, 121 / 135, 131 / 126, 139 / 121, 123 / 132, 133 / 139, 122 / 120,
 * 117 / 120, 127 / 128; at 1536 Q4_K 181 / 190, Q5_K 185 / 195, Q6_K 206 / 184, Q8_0 216 / 177; at 2048 267 / 244,
 * 262 / 260, 273 / 240, 311 / 224, 279 / 254, 305 / 270, 272 / 241, 251 / 222, 261 / 253).
 * Fewer large tiles: the small class, up to a token count per format (small tiles / decode + library, us, at
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
 * The class up to 128 tokens, where half of a 256-token tile is empty: small, whatever the number of tiles (77 tokens 28672 x 4096 large / small: Q4_K
 * 51 / 38, Q5_K 52 / 41, Q6_K 57 / 48; 128 tokens 65536 x 1024 Q4_K 1.26 times, IQ4_XS 1.27, Q3_K 1.30; Q8_0 even). Past 128
 * tokens the class goes by how often the chip has to go round: 256 large tiles (their row tiles are padded to eights) run at a time, 512 small
 * ones, and a small round costs 0.82 of a large one, its last part less the less there is of it (time of small tiles over large,
 * Q4_K ... Q6_K at 4096 columns: one round of large tiles, 512 small ones 0.82 - 0.89, 576 to 768 1.08 - 1.24, 1000 1.24 - 1.37;
 * two rounds, 792 to 960 small ones 0.71 - 0.81, 1160 0.92 - 0.98, 1400 1.06 - 1.14, 1840 1.31 - 1.46; three, 1560 0.81 - 0.87,
 * 2080 1.04 - 1.13, 2800 1.27 - 1.42; Q8_0's small tiles cost 1.2 times as much).
 * Tensors share a launch only if each is of the same class by itself, so the rounds count for those that come with others only
 * where they hold for the company too. Half to twice as many rows as columns (a Q, whose K and V are of the small class): large from
 * 200 on, as for tensors of any size before (Q4_K Q, K and V of 4096 + 1024 + 1024 rows x 4096 at 1280 tokens shared / Q apart in large
 * tiles 80 / 99, 5120 + 1024 + 1024 x 5120 at 1024 97 / 119). More, below eight times (gate and up): by rounds where one tensor and the
 * pair agree, else the same (2 x 10240 x 2560 Q2_K at 984 tokens large / small tiles 117 / 134, 2 x 5888 x 1536 Q4_K at 1440 76 / 81). */
static bool small_by_rounds(uint32_t type, long long n_rows, int n_tok, int n_mat) {
    const long long padded = ((n_rows + 127) / 128 * n_mat + 7) / 8 * 8 * ((n_tok + 255) / 256), rounds = (padded + 255) / 256;
    return (n_rows + 63) / 64 * n_mat * ((n_tok + 127) / 128) <= (rounds == 1 || type == T_Q8_0 ? 512 : 650) * rounds;
}
FusedTile choose_fused_tile(uint32_t type, int n_rows, int n_cols, int n_tok, int ldx, bool have_workspace, bool estimates) {
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
     * and V of a model wider than 11008 divide K at such token counts, and would part from a Q in tiles; past 4096 tokens Q2_K 819 x 1024
     * at 7370 took 42 us in tiles, decode + library 28), and for more rows, where the library's product can be far slower than estimated (24
     * products of 29572 to 44444 rows x 8448 to 14336 at 555 to 1768 tokens: tiles take 0.50 to 0.92 of its time). Rows below 1024 elements, which they were not fitted to, go by them only from
     * decode + library to tiles (Q6_K 1697 x 512 at 1700, the mean of 2400: 0.65 of the time), not between tiles (Q2_K 3048 x 512 at 1816
     * 14.1 -> 16.4). */
    const bool tiles = large_tiles >= 200 ? large_ok : small_ok;
    if (estimates && (!large_ok || !small_ok) && (n_cols >= 1024 || !tiles) && n_rows >= 640 && n_cols <= (type == T_Q8_0 ? 11008 : 14336) &&
        n_tok <= 4096) {
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
 * What a product takes in one piece is what the lines of choose_fused_tile say, without the estimates beyond them: there Q6_K divides where
 * parts gain 13 % on decode + library, and if tiles come close to that, parts are as good or better still (2560 x 10240 at 753 tokens 54.9 /
 * in tiles 60.9, 2916 x 12800 at 616 70 / 74, 2944 x 11776 at 612 66 / 66).
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
        if (choose_fused_tile(type, (int)std::min(q20 * n_cols / 20, (long long)INT_MAX), n_cols, n_tok, ldx, true, false) == tile) return true;
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
 * 557 tokens lost 1 %. Beyond what the estimates were fitted to 8 % are asked for: of 2460 random products there 44 lost more than 3 % and up
 * to 33 with 4 % (Q2_K 2320 x 1536 at 8568 tokens 116 -> 154 us, Q4_K 14892 x 512 at 1540 50 -> 61, Q2_K 85460 x 1280 at 104 42.0 -> 44.8), nine
 * and up to 8 with 8, two with 10, which leaves more alone. */
int choose_token_blocks(uint32_t type, FusedTile tile, int n_mat, const int *n_rows, int n_cols, int n_tok) {
    double us[6];
    tile_us(type, n_mat, n_rows, n_cols, n_tok, us);
    long long rows = 0;
    for (int i = 0; i < n_mat; i++) rows += n_rows[i];
    const bool fitted = n_cols >= 1024 && n_tok <= 4096 && rows <= 28672;
    int best = tile == kFusedLarge ? 5 : 0;
    double best_us = (fitted ? 0.96 : 0.92) * us[best];
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
    const Wave4Call c = {blocks, n_mat, W, X, Y, n_rows, n_cols, n_tok, ldx, ldy, split, stream};
    switch (type) {
    case T_Q4_K: return wave4_q4k(c);
    case T_Q5_K: return wave4_q5k(c);
    case T_Q6_K: return wave4_q6k(c);
    case T_Q8_0: return wave4_q8_0(c);
    case T_IQ4_NL: return wave4_iq4nl(c);
    case T_IQ4_XS: return wave4_iq4xs(c);
    case T_Q4_0: return wave4_q4_0(c);
    case T_Q2_K: return wave4_q2k(c);
    case T_Q3_K: return wave4_q3k(c);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace qlin
