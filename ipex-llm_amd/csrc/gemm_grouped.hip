// Grouped products for mixture-of-experts layers: one launch covers the rows routed to every expert.
//
// The reference has no single call for it: it loops over the experts in Python and calls each expert's
// LowBitLinear on the rows routed to it (python/llm/src/ipex_llm/transformers/models/qwen2_moe.py:375-430
// is the pattern; the gated MLP of an expert is models/common.py:145-158).
//
// Three forms of the tiled MFMA GEMM kernel serve it:
//   - 128-row tiles, two workgroups per compute unit: a group of r rows takes ceil(r / 128) row tiles, each
//     of which walks (loads and dequantizes) the group's weights once;
//   - 256-row tiles ("tall"), one workgroup per compute unit: one walk for up to 256 rows, only the 32-row
//     blocks that hold rows are computed.  With a hundred and more rows per group - a prefill batch spread over
//     the experts - every group above 128 rows would otherwise walk its weights twice.
//   - the narrow tile of the dense GEMM (128 rows by 128 weight rows, one or two groups of waves) where the tiles are few:
//     twice the workgroups of the 128-row form, four times those of the tall one's fused variant.
// The tall form also has the fused gate/up variant (act(x Wg^T) * (x Wu^T) in one pass over x), as has the narrow tile, and can split
// K over a second grid dimension when the output alone has too few tiles for the machine (the down
// projection: few columns, long K); the fp32 partial tiles go through a workspace and a second kernel.
//
// This file: the choice of form and K splits, and the dispatch over the weight formats (instantiated in
// gemm_grouped_<format>.hip from lowbit_gemm_grouped.h).
#include <hip/hip_runtime.h>
#include "lowbit_formats.h"
#include "lowbit_grouped_plan.h"

namespace lowbit {

template <int QT>
int launch_grouped_q(const void *x, const void *const *w, const void *const *w_up, void *y, const int32_t *offsets,
                     int n_groups, int total_rows, int dt, int N, int K, int act, const GroupedPlan &plan, float *ws,
                     hipStream_t st);

template <int QT>
int launch_mlp_gemm_q(const void *x, const void *wg, const void *wu, void *y, int dt, int M, int N, int K, int act,
                      const GroupedPlan &plan, hipStream_t st);

static int device_cus() {
    static const int n_cus = [] {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
            n = 256;
        return n > 0 ? n : 256;
    }();
    return n_cus;
}

// Groups of more than 64 rows on average: how unevenly long they are then decides when a launch ends.
// The routing is not known here, so the order (longest_first) and the cells (tall_chunk) have to be right for any of that average.
// Whole experts over 28 routings each of six blocks (72 to 150 rows a group on average; logits N(0, 1) and, per expert, N(0, s) with s =
// 0, 0.5, 1), against the groups' own order and whole rows, with the sort in one launch and the partial sums' loads at once on top:
// 1.02 to 1.20 times as fast per block with s = 0.5 and 1, 1.00 to 1.03 with s = 0 (1.12 with 32 experts), 12 of 168 slower, 0.977 at
// worst (450 tokens, four of 16 of [6144 x 3072] in asym_int4, groups of 0 to 273 rows).
static bool long_groups(int total_rows, int n_groups) { return total_rows > 64 * n_groups; }

// Column tiles per cell of a plain tall launch: an eighth of a row tile, with long groups a single round of workgroups included.  A
// row tile per XCD keeps its x in one L2, but gives the XCD of the longest group, or of a ninth row tile, twice the others' work
// (512 tokens through two of 8 experts of [14336 x 4096], whole experts, us: fp8_e4m3 528 -> 498, sym_int4 482 -> 468; 600 through
// four of 16 of [4096 x 2048] in sym_int8 241 -> 232; but 200 through two of those 8, 50 rows each, 298 -> 302).
static int tall_chunk(int total_rows, int n_groups, int tiles_n, bool one_round) {
    return grouped_chunk(tiles_n, one_round && !long_groups(total_rows, n_groups));
}

// Bytes of workspace per K split of the tall form: a partial tile per workgroup of the launch, whichever of the two
// tile orders it takes (the grid, and with it a workgroup's slot in the workspace, depends on the order).
static int tall_grid(int total_rows, int n_groups, int tiles_n, bool one_round) {
    return grouped_grid(grouped_max_row_tiles(total_rows, n_groups, G_GM_TALL), tiles_n, tall_chunk(total_rows, n_groups, tiles_n, one_round));
}
static size_t tall_split_bytes(int total_rows, int n_groups, int N) {
    const int tiles_n = (N + G_GN - 1) / G_GN;
    const int a = tall_grid(total_rows, n_groups, tiles_n, false), b = tall_grid(total_rows, n_groups, tiles_n, true);
    return (size_t)(a > b ? a : b) * G_GM_TALL * G_GN * sizeof(float);
}

// Form and K splits for a grouped product given `ws_bytes` of workspace.  Measured on MI355X (8 groups of
// fp8_e4m3 weights, [14336 x 4096] and [4096 x 14336]):
//   - K is split when the tall tiles alone would leave compute units idle: as many splits as it takes for about
//     one workgroup per unit, at most 4, at least 8 K steps each.  With few columns and a long K (the down
//     projection) that beats both unsplit forms at every row count (32 rows per group: 131 against 193 us).
//   - Otherwise the 128-row form with two workgroups per unit is ahead up to about 96 rows per group (147
//     against 156 us at 96) and the tall form from there on (108-150 rows per group: 195 against 245 us).
// Waves per workgroup of the tall form.  Eight (32 weight rows each, two per SIMD) cover part of each other's waits
// where a tile has few MFMAs per weight: measured on MI355X with eight groups of 110-151 rows of fp8_e4m3 weights,
// the fused gate/up launch ([14336 x 4096] twice) takes 341-352 us with eight waves against 372-375 with four; the
// plain product of the down projection ([4096 x 14336], two K splits) 169 against 153-156 - its workgroups are a
// single round, and eight waves read every x operand from LDS twice as often.
static int grouped_waves(int total_rows, int n_groups, bool fused) {
    return fused && (int64_t)total_rows <= (int64_t)n_groups * 192 ? 8 : 4;
}

// Whether the workgroups that hold rows (an estimate: the host never sees the offsets) all run at once: the tall
// form holds one workgroup per compute unit, the 128-row form two.  The tile order then keeps a row tile's column
// tiles on one XCD (see grouped_tile) - when there are row tiles for every XCD.
static bool grouped_one_round(int total_rows, int n_groups, int tiles_n, bool tall, int splits) {
    const int rows = tall ? G_GM_TALL : G_GM_TALL / 2;
    const int row_tiles = total_rows / rows > n_groups ? total_rows / rows : n_groups;
    return row_tiles >= 8 && (int64_t)row_tiles * tiles_n * splits <= (int64_t)device_cus() * (tall ? 1 : 2);
}

// Narrow tiles of a grouped launch: how many groups of waves (0: another form) and the column tiles per cell.
struct NarrowPlan {
    int groups, chunk;
};

// Whether a grouped launch takes narrow tiles (128 rows by 128 weight rows, of both weights 64), and with how many groups of
// waves: 2 while its tiles (an estimate: the host never sees the offsets) are one per CU at most and K has eight steps, 1
// while they are two per CU, 0 beyond.  The fused form's tall tiles are a quarter as many and leave CUs idle there, whole
// experts, us: 15 of [896 x 2048] in nf4 with 114 tokens, two each, 54.9 -> 46.4, 9 of [640 x 1920] in sym_int8 with 93
// tokens, four each, 44.5 -> 39.7, 9 of [1536 x 3968] in sym_int4 with 496 tokens 122.9 -> 109.4; more tiles: 12 of
// [7168 x 2048] in fp8_e4m3 with 300 tokens 169.7 / 178.7, 8 of [14336 x 4096] with 512 492 / 586.
// A group counts as one row tile up to 64 rows on average, else as half a tile more than its rows fill, and as whole tiles at
// least if all have the same (21 of [1872 x 2304] with 2924 tokens in sym_int8 are 630 tiles: 42.8 us in the 128-row form, 66.6 in
// narrow tiles).
// The cells are the largest ones with which no XCD gets more tiles than its CUs hold at once - whole rows of column tiles, an
// eighth, halves of that - because the tiles are about as many as the CUs hold, and a cell more than the others is a second
// round.  A row tile more than the estimate is reckoned with where groups may be uneven.  Whole rows whatever the XCDs' shares,
// as before / now, us: 18 of [720 x 3712] in sym_int8 with 202 tokens, fused, 43.7 / 24.2, 10 of [1088 x 10752] in fp8_e4m3 with
// 178 110 / 69, 18 of [1600 x 1664] in sym_int4 with 179, plain, 21.0 / 13.8, 10 of [6032 x 9856] with 300 203 / 104.
// Random sizes against the forms that narrow tiles replaced: 1.18 times as fast over 2650 fused launches and 1.22 over 4030 plain
// ones; 2 and 1 % of them are slower by more than 4 %, 0.80 and 0.68 at worst: uneven groups whose tiles are more than the
// estimate and than the CUs hold, which are 1.3 times as fast on average all the same.
static NarrowPlan grouped_narrow(int total_rows, int n_groups, int tiles_n, int K) {
    const int rows = G_GM_TALL / 2, cus = device_cus();
    const int uneven = total_rows / rows + (n_groups + 1) / 2, even = (total_rows / n_groups + rows - 1) / rows * n_groups;
    const int row_tiles = total_rows > 64 * n_groups ? (uneven > even ? uneven : even) : n_groups;
    const int64_t tiles = (int64_t)row_tiles * tiles_n;
    if (tiles > 2 * cus) return {0, 0};
    const int groups = tiles <= cus && K / TILE_COLS >= 8 ? 2 : 1, most = cus / 8 * (groups == 2 ? 1 : 2);
    const int unsure = total_rows > 32 * n_groups ? 1 : 0;
    const bool whole = row_tiles >= 8 && grouped_grid(row_tiles + unsure, tiles_n, tiles_n) <= 8 * most;
    int chunk = whole ? tiles_n : (tiles_n + 7) / 8;
    while (chunk > 1 && grouped_grid(row_tiles, tiles_n, chunk) > 8 * most) chunk = (chunk + 1) / 2;
    return {groups, chunk};
}

GroupedPlan grouped_plan(int total_rows, int n_groups, int N, int K, size_t ws_bytes) {
    const int tiles_n = (N + G_GN - 1) / G_GN, G = K / TILE_COLS;
    const int row_tiles = total_rows / G_GM_TALL > n_groups ? total_rows / G_GM_TALL : n_groups;   // estimate of the tiles that hold rows
    int s = device_cus() / (tiles_n * row_tiles);
    s = s > 4 ? 4 : s;
    while (s > 1 && G / s < 8) s--;
    const size_t per_split = tall_split_bytes(total_rows, n_groups, N);
    while (s > 1 && (size_t)s * per_split > ws_bytes) s--;
    if (s < 1) s = 1;
    // Narrow tiles in place of either unsplit form (the same experts, down projection: 54.9 -> 46.9, 44.5 -> 42.4, 122.9 ->
    // 116.4), and of two splits where each tile has a CU and groups are small: the halves of K then meet without a second
    // launch (16 of [2048 x 4096] in nf4 with 300 tokens, two each, 126.0 -> 119.7).
    const NarrowPlan narrow = grouped_narrow(total_rows, n_groups, (N + G_GN / 2 - 1) / (G_GN / 2), K);
    if (s == 1 ? narrow.groups > 0 : s == 2 && narrow.groups == 2 && total_rows <= 96 * n_groups)
        return {false, 1, 4 * narrow.groups, narrow.chunk, narrow.groups};
    const bool tall = s > 1 || (int64_t)total_rows > (int64_t)n_groups * 96;
    const bool one_round = grouped_one_round(total_rows, n_groups, tiles_n, tall, s);
    GroupedPlan plan = {tall, s, grouped_waves(total_rows, n_groups, false), tall ? tall_chunk(total_rows, n_groups, tiles_n, one_round) : grouped_chunk(tiles_n, one_round)};
    plan.longest_first = tall && long_groups(total_rows, n_groups);
    return plan;
}

// Sizes whose tiles (the narrowest: 128 rows by 64 columns) or workgroups 32-bit counts do not hold, or barely: neither planned nor
// launched.
static bool grouped_too_many(int total_rows, int n_groups, int N) {
    return total_rows > 0x7fffff00 || N > 0x7fffff00 || n_groups > (1 << 24) ||
           (int64_t)grouped_max_row_tiles(total_rows, n_groups, G_GM_TALL / 2) * ((N + G_GN / 4 - 1) / (G_GN / 4)) > (1 << 28);
}

// What launch_grouped_gemm would do for a plain grouped product: {tall, splits, waves, grid.x}.  False: it would refuse.
bool grouped_plan_query(int total_rows, int n_groups, int N, int K, size_t ws_bytes, int out[4]) {
    if (grouped_too_many(total_rows, n_groups, N)) return false;
    const GroupedPlan p = grouped_plan(total_rows, n_groups, N, K, ws_bytes);
    const int tiles_n = p.narrow ? (N + G_GN / 2 - 1) / (G_GN / 2) : (N + G_GN - 1) / G_GN;
    out[0] = p.tall;
    out[1] = p.splits;
    out[2] = p.tall || p.narrow ? p.waves : 4;
    out[3] = grouped_grid(grouped_max_row_tiles(total_rows, n_groups, p.tall ? G_GM_TALL : G_GM_TALL / 2), tiles_n, p.chunk);
    return true;
}

size_t grouped_workspace_bytes(int total_rows, int n_groups, int N, int K) {
    if (grouped_too_many(total_rows, n_groups, N)) return 0;
    const GroupedPlan p = grouped_plan(total_rows, n_groups, N, K, (size_t)-1);
    return p.splits > 1 ? (size_t)p.splits * tall_split_bytes(total_rows, n_groups, N) : 0;
}

static GroupedPlan grouped_mlp_plan(int total_rows, int n_groups, int N, int K) {
    const NarrowPlan narrow = grouped_narrow(total_rows, n_groups, (N + G_GN / 4 - 1) / (G_GN / 4), K);
    if (narrow.groups) return {false, 1, 4 * narrow.groups, narrow.chunk, narrow.groups};
    const int tiles_n = (N + G_GN / 2 - 1) / (G_GN / 2);
    GroupedPlan plan = {true, 1, grouped_waves(total_rows, n_groups, true), grouped_chunk(tiles_n, grouped_one_round(total_rows, n_groups, tiles_n, true, 1))};
    plan.longest_first = long_groups(total_rows, n_groups);
    return plan;
}

// y[rows of group e] = x[rows of group e] * dequant(w[e])^T, or, with w_up, act(x w[e]^T) * (x w_up[e]^T).
// workspace (may be null): lets the plain product split K.
int launch_grouped_gemm(const void *x, const void *const *w, const void *const *w_up, void *y, const int32_t *offsets,
                        int n_groups, int total_rows, int qtype, int act_dtype, int N, int K, int act, void *workspace,
                        size_t workspace_bytes, hipStream_t st) {
    if (total_rows == 0 || N == 0 || n_groups == 0) return 0;
    if (total_rows >= (1 << 24) || K >= (1 << 23) || grouped_too_many(total_rows, n_groups, N)) return -3;   // 24-bit row offsets in the kernel
    float *ws = (float *)workspace;
    const GroupedPlan plan = w_up ? grouped_mlp_plan(total_rows, n_groups, N, K)
                                  : grouped_plan(total_rows, n_groups, N, K, ws ? workspace_bytes : 0);
    switch (qtype) {
    case QT_SYM_INT4: return launch_grouped_q<QT_SYM_INT4>(x, w, w_up, y, offsets, n_groups, total_rows, act_dtype, N, K, act, plan, ws, st);
    case QT_ASYM_INT4: return launch_grouped_q<QT_ASYM_INT4>(x, w, w_up, y, offsets, n_groups, total_rows, act_dtype, N, K, act, plan, ws, st);
    case QT_SYM_INT8: return launch_grouped_q<QT_SYM_INT8>(x, w, w_up, y, offsets, n_groups, total_rows, act_dtype, N, K, act, plan, ws, st);
    case QT_NF4: return launch_grouped_q<QT_NF4>(x, w, w_up, y, offsets, n_groups, total_rows, act_dtype, N, K, act, plan, ws, st);
    case QT_FP8_E4M3: return launch_grouped_q<QT_FP8_E4M3>(x, w, w_up, y, offsets, n_groups, total_rows, act_dtype, N, K, act, plan, ws, st);
    default: return -2;
    }
}

// Which tiles a dense gated MLP takes: narrow ones (64 columns of both weights), in halves of 64 rows and with two groups of
// waves, while they are one per CU at most (eight K steps and more); with one group while they are two per CU and M more
// than 128, and where the tall tiles of 256 x 128 would be little more than one per CU, so that most CUs wait for the
// others' second - a last row tile of 64 rows at most is soon done and does not count ([12032 x 5120] at 522 rows in asym_int4
// 137 / 161).  3086 random sizes, M = 65 .. 2048, five formats: 1.84 times as fast as tall tiles alone on average, 0.94 at
// worst.  Tall / narrow, sym_int4 fp16, us:
// [3584 x 1152] at M = 128 / 512 18.1 / 10.8 and 31.6 / 15.8, [8064 x 3840] at M = 128 / 384 43.5 / 25.1 and 77.7 / 54.3,
// [11008 x 4096] at M = 128 / 256 / 768 49.3 / 33.1, 81.2 / 56.4 and 183 / 149; but at M = 512 / 2048 90 / 100 and 319 / 335.
static GroupedPlan mlp_plan(int M, int N, int K) {
    const int rows = G_GM_TALL / 2, tiles_m = (M + rows - 1) / rows, cus = device_cus();
    const int64_t tiles = (int64_t)tiles_m * ((N + G_GN / 4 - 1) / (G_GN / 4));
    const int tall_n = (N + G_GN / 2 - 1) / (G_GN / 2);
    const int64_t tall = (int64_t)((M + G_GM_TALL - 1) / G_GM_TALL) * tall_n, tall_long = (int64_t)((M + G_GM_TALL - 65) / G_GM_TALL) * tall_n;
    GroupedPlan plan = {true, 1, grouped_waves(M, 1, true), grouped_chunk(tall_n, grouped_one_round(M, 1, tall_n, true, 1))};
    if (tiles <= cus && K / TILE_COLS >= 8) plan.narrow = 2;
    else if ((tiles <= 2 * cus && (M > rows || tiles <= cus)) || (tall_long > cus && tall * 20 <= (int64_t)cus * 27)) plan.narrow = 1;
    if (plan.narrow) plan.waves = 4 * plan.narrow;
    plan.halves = plan.narrow && M > rows / 2 && 2 * tiles <= cus;
    return plan;
}

// y = act(x wg^T) * (x wu^T) for a dense gated MLP of M rows: the fused gate/up form of the grouped kernel on one
// group, its weights passed as arguments (nothing is read from tables in device memory).  Measured on MI355X
// against the two products as separate launches plus the activation as an elementwise kernel, sym_int4
// [11008 x 4096] twice: fp16 M = 512 / 2048: 117.5 -> 94.9 / 362.6 -> 318.1 us, bf16 137.2 -> 94.3 / 401.6 -> 316.6;
// nf4 [28672 x 8192] bf16 at M = 256 / 1024: 354.8 -> 233.6 / 1008 -> 892.
int launch_mlp_gemm(const void *x, const void *wg, const void *wu, void *y, int qtype, int act_dtype, int M, int N, int K,
                    int act, hipStream_t st) {
    if (M == 0 || N == 0) return 0;
    if (M >= (1 << 24) || K >= (1 << 23)) return -3;                 // 24-bit row offsets in the kernel
    const GroupedPlan plan = mlp_plan(M, N, K);
    switch (qtype) {
    case QT_SYM_INT4: return launch_mlp_gemm_q<QT_SYM_INT4>(x, wg, wu, y, act_dtype, M, N, K, act, plan, st);
    case QT_ASYM_INT4: return launch_mlp_gemm_q<QT_ASYM_INT4>(x, wg, wu, y, act_dtype, M, N, K, act, plan, st);
    case QT_SYM_INT8: return launch_mlp_gemm_q<QT_SYM_INT8>(x, wg, wu, y, act_dtype, M, N, K, act, plan, st);
    case QT_NF4: return launch_mlp_gemm_q<QT_NF4>(x, wg, wu, y, act_dtype, M, N, K, act, plan, st);
    case QT_FP8_E4M3: return launch_mlp_gemm_q<QT_FP8_E4M3>(x, wg, wu, y, act_dtype, M, N, K, act, plan, st);
    default: return -2;
    }
}

}  // namespace lowbit
