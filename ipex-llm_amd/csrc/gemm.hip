// Prefill product y[M,N] = x[M,K] * dequant(W)[N,K]^T for large M (compute-bound).
//
// Replaces xe_linear.forward_new at large M
// (python/llm/src/ipex_llm/transformers/low_bit_linear.py:660-668).
//
// Workgroup tile: 128 rows of x (M) by 256 weight rows (N), 4 waves side by side along N,
// so that every weight is dequantized by exactly one wave.  Per 128-column step of K:
//   weights: each lane loads its 16/32 bytes of four tiles straight from HBM into registers -
//            the tiled layout already is the MFMA operand layout - and turns them into scaled
//            fp16 / bf16 values in registers (no LDS for weights);
//   x:       the workgroup copies the 128 x 128 block of x into LDS in operand order
//            (double buffered), and every wave reads it from there;
//   8 v_mfma_f32_32x32x16 per 16 columns and wave, weights as the A operand (rows = n) and x
//   as the B operand (columns = m), so a lane ends up with groups of 4 consecutive n for one m
//   and stores 8 contiguous bytes of y at a time.
// FLOP per launch: 2*M*N*K; MFMA-bound (fp16 / bf16 dense peak).
#include "lowbit_gemm_kernel.h"
#include "lowbit_splits.h"

namespace lowbit {

int launch_gemv(const void *x, const void *w, const void *bias, void *y, int qtype, int layout, int act_dtype, int M, int N, int K,
                int waves, hipStream_t st);

int launch_gemm_rows(const void *x, const void *w, const void *bias, void *y, int qtype, int act_dtype, int M, int N, int K,
                     void *workspace, size_t workspace_bytes, hipStream_t st);

// Sums the fp32 partial tiles of the splits (stored in the GEMM's register layout: split, tile, wave,
// register group, lane) and writes y, rounded once.  One thread per group of 4 consecutive n.
template <typename AT>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float *__restrict__ ws, AT *__restrict__ y,
                                                            const AT *__restrict__ bias, int M, int N, int splits, int tile_rows) {
    const int tiles_n = (N + GN - 1) / GN;
    const int64_t n_tiles_all = (int64_t)((M + tile_rows - 1) / tile_rows) * tiles_n;
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;       // (tile, wave, group, lane): a block's groups are of one wave
    constexpr int BLOCKS = MB32 * NB32 * 4 / 4;                      // blocks of threads per wave
    const int lane = threadIdx.x & 63, grp = (int)(blockIdx.x % BLOCKS) * 4 + (threadIdx.x >> 6);
    const int wave = (int)(blockIdx.x / BLOCKS % 4), tile_id = (int)(blockIdx.x / (4 * BLOCKS));
    const int mb = grp / (NB32 * 4), nb = grp / 4 % NB32, q = grp % 4;
    const int m = tile_id / tiles_n * tile_rows + mb * 32 + (lane & 31);
    const int n = tile_id % tiles_n * GN + wave * GN_WAVE + nb * 32 + q * 8 + (lane >> 5) * 4;
    if (mb * 32 >= tile_rows || m >= M || n >= N) return;
    const int64_t per_split = n_tiles_all * 4 * (MB32 * NB32 * 4) * 64 * 4;     // floats
    const f32x4 a = sum_splits((const f32x4 *)ws + t, per_split / 4, splits);
    typedef AT at4 __attribute__((ext_vector_type(4)));
    at4 o;
#pragma unroll
    for (int k = 0; k < 4; k++) o[k] = to_at<AT>(bias ? a[k] + (float)bias[n + k] : a[k]);
    *(at4 *)(y + (int64_t)m * N + n) = o;
}

// A launch of the 128-row DMA form whose tiles leave most compute units idle goes out in half tiles of 64 rows, twice
// as many workgroups (see the kernel).  Half a tile pays the whole tile's dequantization and takes three quarters of
// its time per K step.  Measured on sym_int4 fp16 without a workspace, each launch on weights it has not just read:
// [4096 x 4096] at M = 128 / 512 / 768 (16 / 64 / 96 tiles): 38.9 -> 31.6 / 41.3 -> 34.1 / 41.7 -> 37.4 us;
// [11008 x 4096] at M = 128 / 256 (43 / 86 tiles): 40.3 -> 33.9 / 41.3 -> 35.8 us; [4096 x 11008] at M = 512:
// 99.4 -> 82.7 us.  At 112-128 tiles the two are level, and as soon as two halves share a unit it loses: 129 tiles
// 47 -> 57 us, 256 tiles ([4096 x 4096] at M = 2048) 64 -> 75 us.  Cutting only the tiles of a large launch's last,
// partly filled round changes nothing (688 tiles: 161 us either way) or loses 2-6 %.
static bool half_tiles(int M, int64_t tiles, int n_cus) { return M > GM / 2 && tiles * 8 <= (int64_t)n_cus * 3; }

// Estimated run time in microseconds of the 128-row GEMM with K split `splits` ways (1 = no split), fitted to
// measurements on MI355X: 40 weight shapes from [1024 x 8192] to [28672 x 8192] in all five formats, M = 17 .. 768,
// 1 .. 16 splits, each launch on weights it has not just read (6200 launches; 9.6 % rms).  What the fit holds:
//   - a 128-column step takes a workgroup 1.2 us while the launch has up to 128 workgroups, 1.5 us at one per CU,
//     and 2.1 us and more as soon as two share a CU - a launch of 258 workgroups takes as long as its two shared
//     CUs ([11008 x 4096] at M = 256: 2 splits = 172 workgroups 36.7 us, 3 splits = 258 workgroups 45.9 us), so the
//     splits that pay keep the workgroups at or below the number of CUs;
//   - a row tile that is partly empty skips the MFMAs of its empty 32-row blocks (a sixth of the step per quarter);
//   - launch, prologue and epilogue come to 2 us, the second launch of a split to 5.4 us, a workgroup's fp32 partial
//     tile to 0.043 us to write and sum (a quarter of it fixed, the rest by the rows it holds);
//   - the formats with more work per weight take longer per step: sym_int8 1.30, fp8_e4m3 1.15, nf4 1.30 - 2.48 in
//     the register-staged form it uses up to one workgroup per CU; half tiles take 0.88 (0.83) of a tile's step.
// (abi.hip's one_pass_applies has a fit of its own on top of this, to be made again when this changes.)
double gemm_time_us(int M, int N, int K, int splits, int qtype) {
    const int tiles_m = (M + GM - 1) / GM;
    const double tiles = (double)tiles_m * (double)((N + GN - 1) / GN);
    const int G = K / TILE_COLS;
    const int k_steps = (G + splits - 1) / splits;
    const int ny = (G + k_steps - 1) / k_steps;
    const bool halves = ny == 1 && qtype != QT_NF4 && half_tiles(M, (int64_t)tiles, 256);   // (nf4: register-staged form)
    const double wgs = tiles * ny * (halves ? 2.0 : 1.0);
    const bool heavy = qtype == QT_SYM_INT8 || qtype == QT_FP8_E4M3;
    const double format = qtype == QT_NF4 ? (wgs <= 256.0 ? 2.48 : 1.30) : qtype == QT_SYM_INT8 ? 1.30 : qtype == QT_FP8_E4M3 ? 1.15 : 1.0;
    const double half = !halves ? 1.0 : heavy ? 0.83 : 0.88;
    const double over128 = wgs > 128.0 ? (wgs - 128.0) / 128.0 : 0.0;
    const double step = wgs <= 256.0 ? 1.21 + 0.29 * over128 : 2.12 + 0.56 * ((wgs < 512.0 ? wgs : 512.0) - 256.0) / 256.0;
    // workgroups beyond two per CU wait for a slot: the launch lasts as long as the CU that gets most of them
    const double rounds = wgs > 512.0 ? (double)(((int64_t)wgs + 255) / 256) / 2.0 : 1.0;
    const double fill = (double)M / ((double)tiles_m * GM);
    double t = 2.1 + (double)k_steps * step * format * half * rounds * (0.83 + 0.17 * fill);
    if (ny > 1) t += 5.4 + 0.043 * (double)ny * tiles * (0.24 + 0.76 * fill);
    return t;
}

// Number of K splits to use for this shape given `ws_bytes` of workspace (1 = none): the fastest by the estimate
// above among 1 .. 16 splits of at least two K steps that fit the workspace.  On the shapes the estimate was fitted
// to, the split it picks is within 2 % of the best measured one on average.
int gemm_splits(int M, int N, int K, size_t ws_bytes, int qtype) {
    const size_t tiles = (size_t)((M + GM - 1) / GM) * (size_t)((N + GN - 1) / GN);
    const size_t per_split = tiles * GM * GN * sizeof(float);     // whole tiles: partial sums keep the tile layout
    const int G = K / TILE_COLS;
    int best = 1;
    double best_t = gemm_time_us(M, N, K, 1, qtype);
    for (int s = 2; s <= 16 && s * 2 <= G; s++) {
        if ((size_t)s * per_split > ws_bytes) break;
        const double t = gemm_time_us(M, N, K, s, qtype);
        if (t < best_t) {
            best = s;
            best_t = t;
        }
    }
    return best;
}

// How many column tiles (256 weight rows each) the tall form takes, from the left; the 128-row form covers the columns that are
// left.  0 = the tall form is not used: a last row tile that is less than half full (the 128-row form computes 128 rows less), K too
// long for 24-bit row offsets, or one of the rules below.  A launch of tall tiles takes 3.3 us per K step and whole round of one
// tile per CU and 1.75 + 1.3 f for a round of which a part f is filled (fewer CUs at work run faster), 8 us per round: fitted to 500
// random sizes, M = 140 .. 2048, five formats, both types, 3 % rms in each.  Hence
//   - all columns in up to one round, from 0.52 of it on and where 128-row tiles would be more than one per CU ([12288 x 4096] at M =
//     700 in nf4 118 -> 83 us, at M = 1000 in bf16 sym_int4 114 -> 95, in fp16 100 -> 95; 0.4 to 0.5 of a round 1.2 times the time);
//   - all columns where the last round is whole or half full at least (0.65 of it in fp16 and 4-bit integers, which cost the 128-row
//     form least), from 8 steps on ([28672 x 8192] at M = 1000, 1.75 rounds: nf4 431 -> 403 us, bf16 sym_int4 435 -> 393, fp16 402 ->
//     386, fp8_e4m3 404 -> 385);
//   - else whole rounds, so that no CU sits idle while another works on one more tall tile, where the rest costs less than they gain:
//     fp8_e4m3 and 4-bit integers in bf16 from 16 steps on ([12288 x 4096] at M = 1500 in bf16 sym_int4 168 -> 157; fewer steps lose
//     up to 16 %).  None of the 500 sizes is slower by more than 2 % with these three than without, and the 180 that they change are
//     1.07 times as fast;
//   - sym_int8 and nf4 pay most per weight for the dequantization, which the tall form does half as often: the estimate
//     of gemm_time_us for both ways, 0.9 of a full 128-row round for a tall one, nf4's remainder, in narrow tiles, 1.15
//     (sym_int8 [28672 x 8192] at M = 700 347 us without tall tiles and 332 with; nf4 there 404 and 328, [11008 x 4096] at
//     M = 2047 207 and 171; [11008 x 4096] at M = 1300, 258 tall tiles, one column left over: 116 us without, 151 with);
//   - the others with 1.5 workgroups per CU left over (at M = 2048 on [11008 x 4096] sym_int4 +1 %, fp8_e4m3 -3 %).
static double steps_time(int64_t wgs) {                  // a 128-column step of the 128-row form, see gemm_time_us
    if (wgs > 512) return 2.68 * (double)((wgs + 255) / 256) / 2.0;
    return wgs > 256 ? 2.12 + 0.56 * (double)(wgs - 256) / 256.0 : 1.21 + (wgs > 128 ? 0.29 * (double)(wgs - 128) / 128.0 : 0.0);
}
static bool tall_fits(int M, int K) {
    const int rest = M % GM_TALL;
    return M >= GM_TALL && !(rest && rest <= GM) && M < (1 << 24) && K < (1 << 23);
}
// by the first three rules, 0: none of them
static int tall_by_rounds(int M, int N, int K, int n_cus, int qtype, bool f16) {
    if (!tall_fits(M, K)) return 0;
    const int tiles_m = (M + GM_TALL - 1) / GM_TALL, tiles_n = (N + GN - 1) / GN;
    const int64_t tiles = (int64_t)tiles_m * tiles_n, small = (int64_t)((M + GM - 1) / GM) * tiles_n;
    if (tiles <= n_cus) return small > n_cus && tiles * 100 >= (int64_t)n_cus * 52 ? tiles_n : 0;
    const bool int4 = qtype == QT_SYM_INT4 || qtype == QT_ASYM_INT4;
    const int64_t last = tiles % n_cus;
    if (last == 0 || (last * 100 >= (int64_t)n_cus * (int4 && f16 ? 65 : 50) && K >= 8 * TILE_COLS)) return tiles_n;
    return ((int4 && !f16) || qtype == QT_FP8_E4M3) && K >= 16 * TILE_COLS ? (int)(tiles / n_cus * n_cus / tiles_m) : 0;
}
static int tall_columns(int M, int N, int K, int n_cus, int qtype, bool f16) {
    if (const int cols = tall_by_rounds(M, N, K, n_cus, qtype, f16)) return cols;
    if (M < 2 * GM_TALL || !tall_fits(M, K)) return 0;
    const int tiles_m = (M + GM_TALL - 1) / GM_TALL, tiles_n = (N + GN - 1) / GN;
    const int64_t small_m = (M + GM - 1) / GM;           // row tiles of the 128-row form
    const int rounds = (int)((int64_t)tiles_m * tiles_n / n_cus);
    if (rounds < 1) return 0;
    const int cols = (int)((int64_t)rounds * n_cus / tiles_m);
    if (cols >= tiles_n) return tiles_n;
    const int64_t left = (tiles_n - cols) * small_m;
    if (qtype == QT_SYM_INT8 || qtype == QT_NF4)
        return rounds * 0.9 * 2.68 + steps_time(left) * (qtype == QT_NF4 ? 1.15 : 1.0) < 0.98 * steps_time(tiles_n * small_m) ? cols : 0;
    return 2 * left >= 3 * n_cus ? cols : 0;
}

static int gemm_cus() {
    static const int n_cus = [] {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
            n = 256;
        return n > 0 ? n : 256;
    }();
    return n_cus;
}

// Whether lowbit_linear takes tall tiles whatever the estimates of the other kernels say.
bool gemm_prefers_tall(int qtype, int act_dtype, int M, int N, int K) {
    return tall_by_rounds(M, N, K, gemm_cus(), qtype, act_dtype == DT_F16) > 0;
}

// How many tiles at the end of each XCD's share of a 128-row launch go out as two half tiles: all of them or none.
static int split_tail_tiles(int M, int64_t tiles, int n_cus) {
    return half_tiles(M, tiles, n_cus) ? (int)(tiles / 8) + 1 : 0;
}

template <int QT, typename AT>
static int launch_gemm_t(const void *x, const void *w, const void *bias, void *y, int M, int N, int K, float *ws, int splits,
                         hipStream_t st) {
    if (splits <= 1) ws = nullptr;
    const int G = K / TILE_COLS;
    const int tiles_n_all = (N + GN - 1) / GN;
    const int n_cus = gemm_cus();
    // tall form on the left columns, 128-row form on the rest (both in the same stream, the second starts when
    // the tall tiles, which all take the same time, are done)
    GroupArgs ga{};
    ga.bias = bias;
    const int tall = ws ? 0 : tall_columns(M, N, K, n_cus, QT, __is_same(AT, _Float16));
    if (tall > 0) {
        const int tiles_m = (M + GM_TALL - 1) / GM_TALL;
        ga.tile_rows = GM_TALL;
        ga.row_tiles = tiles_m;
        const unsigned grid = 8 * (unsigned)(((int64_t)tiles_m * tall + 7) / 8);
        // (four waves, which read each x operand from LDS once per two MFMAs: 2-4 % faster than eight)
        hipLaunchKernelGGL((gemm_mfma_kernel<QT, AT, true, MB32_TALL>), dim3(grid), dim3(256), 0, st,
                           (const AT *)x, (const uint8_t *)w, (AT *)y, M, N, K, band_rows(tiles_m), ga, G, (float *)nullptr, 0, tall);
        if (tall == tiles_n_all) return 0;
        if constexpr (QT == QT_NF4) {
            // what is left of nf4 in narrow tiles, which look up in registers too (768 of them: [28672 x 8192] at
            // M = 1000 483 -> 469 us; where at most one 128 x 256 tile per CU is left, which would take the
            // register-staged form below, [11008 x 4096] at M = 2047 212 -> 171, [28672 x 8192] at M = 700 404 -> 328)
            const int left = (N + GN / 2 - 1) / (GN / 2) - 2 * tall, tiles_m = (M + GM - 1) / GM;
            ga.tile_rows = GM;
            ga.row_tiles = tiles_m;
            narrow_form(false, three_blocks(M, GM), [&](auto, auto three) {
                hipLaunchKernelGGL((gemm_mfma_kernel<QT, AT, true, MB32, false, false, 4, true, 1, decltype(three)::value>),
                                   dim3(8 * (unsigned)(((int64_t)tiles_m * left + 7) / 8)), dim3(256), 0, st, (const AT *)x, (const uint8_t *)w,
                                   (AT *)y, M, N, K, band_rows(tiles_m), ga, G, (float *)nullptr, 2 * tall, left);
            });
            return 0;
        }
    }
    const int tn0 = tall, tiles_n = tiles_n_all - tall;
    const int tiles_m = (M + GM - 1) / GM;
    const int band_m = band_rows(tiles_m);
    const int k_steps = ws ? (G + splits - 1) / splits : G;
    const int ny = ws ? (G + k_steps - 1) / k_steps : 1;             // splits that actually hold steps
    const bool fits24 = M < (1 << 24) && K < (1 << 23);              // 24-bit row offsets
    const bool dma = fits24 && (QT != QT_NF4 || tiles_m * tiles_n * ny > 256);
    ga.split_tail = (dma && !ws) ? split_tail_tiles(M, (int64_t)tiles_m * tiles_n, n_cus) : 0;
    ga.tile_rows = dma && !ga.split_tail ? dense_tile_rows(M) : GM;
    ga.row_tiles = tiles_m;
    dim3 grid(8 * (unsigned)(((int64_t)tiles_m * tiles_n + 7) / 8 + ga.split_tail), ny);
    // Two forms of the kernel.  The DMA form (x straight into LDS, one K step of prefetch, 128 vector registers)
    // lets a CU hold two workgroups that cover each other's waits, and is 4-8 % ahead with a single workgroup per
    // CU as well - except with nf4, whose code book reads compete with the DMA for LDS: there the register-staged
    // form with its deeper prefetch is 4 % faster while there is at most one workgroup per CU.
    if (dma && !ga.split_tail && three_blocks(M, ga.tile_rows))
        hipLaunchKernelGGL((gemm_mfma_kernel<QT, AT, true, MB32, false, false, 4, false, 1, true>), grid, dim3(256), 0, st, (const AT *)x,
                           (const uint8_t *)w, (AT *)y, M, N, K, band_m, ga, k_steps, ws, tn0, tiles_n);
    else if (dma)
        hipLaunchKernelGGL((gemm_mfma_kernel<QT, AT, true, MB32>), grid, dim3(256), 0, st, (const AT *)x, (const uint8_t *)w,
                           (AT *)y, M, N, K, band_m, ga, k_steps, ws, tn0, tiles_n);
    else
        hipLaunchKernelGGL((gemm_mfma_kernel<QT, AT, false, MB32>), grid, dim3(256), 0, st, (const AT *)x, (const uint8_t *)w,
                           (AT *)y, M, N, K, band_m, ga, k_steps, ws, tn0, tiles_n);
    if (ws) {
        const int64_t threads = (int64_t)tiles_m * tiles_n * (GM * GN / 4);
        hipLaunchKernelGGL((splitk_reduce_kernel<AT>), dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, st, ws,
                           (AT *)y, (const AT *)bias, M, N, ny, ga.tile_rows);
    }
    return 0;
}

// Whether a launch of narrow tiles goes out in half tiles of 64 rows: while the halves are no more than one per CU.
bool narrow_halves(int M, int N) {
    const int64_t tiles = (int64_t)((M + GM - 1) / GM) * ((N + GN / 2 - 1) / (GN / 2));
    return M > GM / 2 && tiles * 2 <= 256;
}

static int64_t narrow_workgroups(int M, int N) {
    const int64_t tiles = (int64_t)((M + GM - 1) / GM) * ((N + GN / 2 - 1) / (GN / 2));
    return narrow_halves(M, N) ? 2 * tiles : tiles;
}

// Whether a launch of narrow tiles takes two groups of waves per workgroup, each on one half of K (KS in the kernel): as
// long as a CU has one workgroup and K eight steps.  One wave per SIMD cannot cover its own loads and dequantization; two
// workgroups per CU do that for each other, and there the form loses what its sums cost at the end.  One group / two:
// [2048 x 2048] at M = 256 16.4 / 13.6 us in sym_int4 fp16, 17.8 / 15.0 in nf4 bf16, [4096 x 4096] at M = 512 31.4 / 27.3
// and 36.0 / 29.7, [12288 x 4096] at M = 256 40.1 / 33.7 and 42.2 / 37.6; [1024 x 1024], eight steps, at M = 128 / 512
// 8.5 / 8.1 and 10.3 / 9.4; 344 workgroups ([11008 x 4096] at M = 512) 56.0 / 65.2.
static bool narrow_two_groups(int M, int N, int K) { return narrow_workgroups(M, N) <= 256 && K / TILE_COLS >= 8; }

// Estimated run time in microseconds of the narrow form, fitted like gemm_time_us (760 launches, 8.5 % rms): a
// 128-column step takes a workgroup 1.05 us up to 128 workgroups, 1.24 at one per CU, 1.55 - 1.96 once two share a
// CU; half tiles 0.87 of it.  nf4 1.06 with its lookups in registers (80 points, 8 shapes: the choice made with it is
// 1.5 % above the faster of this form and the rest on average; 14 % at worst, [8192 x 8192] at M = 1300);
// the entry points whose choices lowbit_forward_plan reports keep the figure from before, 1.24.
// Two groups of waves (lowbit_linear's estimate only): 888 launches, 6.8 % rms; a pair of steps takes 1.49 us, a million
// weights 0.12 us; scaled by 0.91, in the 8-bit formats by 0.955 (4900 points on weights that were not just read: chosen within
// 1.3 % of the faster way on average as with 0.91, but 96 of them 5 % slower than the other way where it were 271).  Never above the estimate of one group, which two groups did not exceed at any of 2500
// random points: the fit is too long for wide weights of few steps ([26304 x 2432] at 88 rows in sym_int4 26.1 us; where it
// passed them over, 37.6).  Against the choice with one group the one made with this is 6.2 % faster on average over 2164
// of them; 20 are slower by 3 to 11 % (a larger scale loses as much elsewhere).
// (abi.hip's one_pass_applies has a fit of its own on top of this, to be made again when this changes.)
double narrow_time_us(int M, int N, int K, int qtype, bool linear) {
    const int tiles_m = (M + GM - 1) / GM;
    const bool halves = narrow_halves(M, N);
    const double wgs = (double)narrow_workgroups(M, N);
    const double format = qtype == QT_NF4 ? (linear ? 1.06 : 1.24) : qtype == QT_SYM_INT8 ? 1.11 : qtype == QT_FP8_E4M3 ? 1.05 : 1.0;
    const double over128 = wgs > 128.0 ? (wgs - 128.0) / 128.0 : 0.0;
    const double step = wgs <= 256.0 ? 1.05 + 0.20 * over128 : 1.55 + 0.41 * ((wgs < 512.0 ? wgs : 512.0) - 256.0) / 256.0;
    const double rounds = wgs > 512.0 ? (double)(((int64_t)wgs + 255) / 256) / 2.0 : 1.0;
    const double fill = (double)M / ((double)tiles_m * GM);
    const double one = 0.5 + (double)(K / TILE_COLS) * step * format * rounds * (halves ? 0.87 : 1.0) * (0.84 + 0.16 * fill);
    if (!linear || !narrow_two_groups(M, N, K)) return one;
    const double format2 = qtype == QT_NF4 ? 1.12 : qtype == QT_SYM_INT8 ? 1.16 : qtype == QT_FP8_E4M3 ? 1.14 : 1.0;
    const double two = (qtype == QT_SYM_INT8 || qtype == QT_FP8_E4M3 ? 0.955 : 0.91) *
                       (3.86 + 0.97 * over128 + 0.123e-6 * (double)N * (double)K +
                                (double)((K / TILE_COLS + 1) / 2) * 1.485 * format2 * (1.0 + 0.17 * over128) * (halves ? 0.79 : 1.0) * (0.69 + 0.31 * fill));
    return two < one ? two : one;
}

// The narrow form of the 128-row DMA kernel: tiles of 128 x 128, or 64 x 128 (narrow_halves).
template <int QT, typename AT>
static int launch_gemm_narrow_t(const void *x, const void *w, const void *bias, void *y, int M, int N, int K, hipStream_t st) {
    if (M >= (1 << 24) || K >= (1 << 23)) return -3;                 // 24-bit row offsets
    const int G = K / TILE_COLS;
    const int tiles_n = (N + GN / 2 - 1) / (GN / 2), tiles_m = (M + GM - 1) / GM;
    const bool halves = narrow_halves(M, N);
    GroupArgs ga{};
    ga.bias = bias;
    ga.split_tail = halves ? (int)(((int64_t)tiles_m * tiles_n) / 8) + 1 : 0;
    ga.tile_rows = halves ? GM : dense_tile_rows(M);
    ga.row_tiles = tiles_m;
    dim3 grid(8 * (unsigned)(((int64_t)tiles_m * tiles_n + 7) / 8 + ga.split_tail), 1);
    auto launch = [&](auto groups, auto three) {
        constexpr int KS = decltype(groups)::value;
        hipLaunchKernelGGL((gemm_mfma_kernel<QT, AT, true, MB32, false, false, 4, true, KS, decltype(three)::value>), grid, dim3(256 * KS), 0, st,
                           (const AT *)x, (const uint8_t *)w, (AT *)y, M, N, K, band_rows(tiles_m), ga, G, (float *)nullptr, 0, tiles_n);
    };
    narrow_form(narrow_two_groups(M, N, K), !halves && three_blocks(M, ga.tile_rows), launch);
    return 0;
}

template <int QT>
static int launch_gemm_narrow_q(const void *x, const void *w, const void *bias, void *y, int dt, int M, int N, int K, hipStream_t st) {
    if (dt == DT_F16) return launch_gemm_narrow_t<QT, _Float16>(x, w, bias, y, M, N, K, st);
    if (dt == DT_BF16) return launch_gemm_narrow_t<QT, __bf16>(x, w, bias, y, M, N, K, st);
    return -4;
}

int launch_gemm_narrow(const void *x, const void *w, const void *bias, void *y, int qtype, int act_dtype, int M, int N, int K, hipStream_t st) {
    if (M == 0 || N == 0) return 0;
    switch (qtype) {
    case QT_SYM_INT4: return launch_gemm_narrow_q<QT_SYM_INT4>(x, w, bias, y, act_dtype, M, N, K, st);
    case QT_ASYM_INT4: return launch_gemm_narrow_q<QT_ASYM_INT4>(x, w, bias, y, act_dtype, M, N, K, st);
    case QT_SYM_INT8: return launch_gemm_narrow_q<QT_SYM_INT8>(x, w, bias, y, act_dtype, M, N, K, st);
    case QT_NF4: return launch_gemm_narrow_q<QT_NF4>(x, w, bias, y, act_dtype, M, N, K, st);
    case QT_FP8_E4M3: return launch_gemm_narrow_q<QT_FP8_E4M3>(x, w, bias, y, act_dtype, M, N, K, st);
    default: return -2;
    }
}

template <int QT>
static int launch_gemm_q(const void *x, const void *w, const void *bias, void *y, int dt, int M, int N, int K, float *ws, int splits,
                         hipStream_t st) {
    if (dt == DT_F16) return launch_gemm_t<QT, _Float16>(x, w, bias, y, M, N, K, ws, splits, st);
    if (dt == DT_BF16) return launch_gemm_t<QT, __bf16>(x, w, bias, y, M, N, K, ws, splits, st);
    return -4;
}

// splits: 0 = chosen here from the workspace size, otherwise as given (the caller has checked that it fits)
int launch_gemm(const void *x, const void *w, const void *bias, void *y, int qtype, int layout, int act_dtype, int M, int N, int K,
                void *workspace, size_t workspace_bytes, int want_splits, hipStream_t st) {
    if (M == 0 || N == 0) return 0;
    // the MFMA GEMM reads the tiled layout and stores 8-byte groups of y (N % 4 == 0 is implied
    // by N % 16 == 0); row-major weights have their own, a y of another alignment goes through the streaming kernel
    if (layout == LAYOUT_GGML) return launch_gemm_rows(x, w, bias, y, qtype, act_dtype, M, N, K, workspace, workspace_bytes, st);
    if (layout != LAYOUT_TILED || (N % TILE_ROWS) || (K % TILE_COLS) || (((uintptr_t)y) & 7))
        return launch_gemv(x, w, bias, y, qtype, layout, act_dtype, M, N, K, 0, st);
    float *ws = (float *)workspace;
    const int splits = !ws ? 1 : want_splits > 0 ? want_splits : gemm_splits(M, N, K, workspace_bytes, qtype);
    switch (qtype) {
    case QT_SYM_INT4: return launch_gemm_q<QT_SYM_INT4>(x, w, bias, y, act_dtype, M, N, K, ws, splits, st);
    case QT_ASYM_INT4: return launch_gemm_q<QT_ASYM_INT4>(x, w, bias, y, act_dtype, M, N, K, ws, splits, st);
    case QT_SYM_INT8: return launch_gemm_q<QT_SYM_INT8>(x, w, bias, y, act_dtype, M, N, K, ws, splits, st);
    case QT_NF4: return launch_gemm_q<QT_NF4>(x, w, bias, y, act_dtype, M, N, K, ws, splits, st);
    case QT_FP8_E4M3: return launch_gemm_q<QT_FP8_E4M3>(x, w, bias, y, act_dtype, M, N, K, ws, splits, st);
    default: return -2;
    }
}

}  // namespace lowbit
