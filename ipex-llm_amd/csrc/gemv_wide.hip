// Where the one-pass kernel (lowbit_gemv_wide.h) is used, for up to 64 rows of x and for more on small weights, and in which shape.
#include <hip/hip_runtime.h>
#include "lowbit_wide_plan.h"

namespace lowbit {

template <int QT>
int launch_wide_q(const void *x, const void *w, const void *bias, void *y, int layout, int dt, int M, int N, int K, const WideShape &s,
                  hipStream_t st);
template <int QT>
int launch_wide_mlp_q(const void *x, const void *wg, const void *wu, void *y, int dt, int M, int N, int K, int act, const WideShape &s,
                      hipStream_t st);

// The shape for M rows of x, r = 0: another kernel is the faster one.  T tile rows, G column groups, MB 16-row blocks of x;
// measured on MI355X over some 900 points (format, shape, M, activation type, layout), each launch on weights not just read.
//
// R = ceil(T / 256) tile rows a workgroup: one workgroup per CU then covers the weight, and a larger R only makes fewer
// workgroups read the same x.  8 waves (12 where a wave holds one tile and 16 rows, at the latency of the walk; 4 where
// R = 4 and several workgroups share a CU).
// Every workgroup reads all of x from L2, MB * G * 4 KB: beyond about 0.8 MB (MB * G = 192) the ring kernel and the K splits
// of the tiled GEMM win, which divide x as well ([4096 x 11008] at 64 rows: 24.2 us against 31).  Beyond 1024 tile rows
// there are several rounds of workgroups and x comes again in each: only up to 32 rows still pay ([28672 x 8192] at 48
// rows 106 against 96 us of the GEMM).
// linear: lowbit_linear and float32 activations.  The other entry points, whose kernel a caller may rely on, keep the streaming kernel up to 8
// rows of tiled weights (4 of row-major ones) and beyond 1024 tile rows.
static WideShape wide_shape(int qtype, int layout, int dt, int M, int N, int K, bool linear) {
    const int T = (N + TILE_ROWS - 1) / TILE_ROWS, G = (K + TILE_COLS - 1) / TILE_COLS, MB = (M + 15) / 16;
    const int rounds = (T + 255) / 256;
    const WideShape none = {0, 0};
    // 5 .. 8 rows of x and a weight that three tile rows a workgroup cover in one round, where the streaming kernel's workgroups of
    // one or two read x more often: from 24 groups on (8 rows, 16-bit activations: 0.79 .. 0.95 of its time on 9728 .. 12288 rows
    // of 4096 and 8192 columns, sym_int8 on [11008 x 4096] 14.2 -> 11.3 us, asym_int4 in bf16 10.9 -> 9.2, float32 sym_int4 15.2 -> 12.8;
    // 1.0 .. 1.07 of it with 8 groups).
    const bool shared_by_three = linear && M > 4 && M <= 8 && layout == LAYOUT_TILED && rounds == 3 && G >= 24;
    if (dt == DT_F32) {
        // Two planes of x: 32 rows at most, and twice the x to read, to split and to write to LDS.  One pass at half the x traffic of
        // the streaming kernel's (9 .. 16 rows on [28672 x 8192]: 86 -> 48) or in place of two; up to 8 rows it loses.
        // As few workgroups as cover the weight in one round, as with 16-bit activations, now that splitting x is short enough for
        // x to be shared by three tile rows (two, in two rounds, before): 9 / 24 rows on [11008 x 4096] in sym_int4 18.6 -> 12.8
        // / 30.4 -> 17.7 us, on [9600 x 8192] 31.7 -> 19.6 / 55.3 -> 29.6.  Four tile rows have the registers for 16 rows
        // of x only, and row-major weights need more instructions per tile: [14336 x 4096], 9 rows, four / two tile rows 15.2 / 17.2
        // us.  Beyond 1024 tile rows three with four waves, several workgroups per CU ([18000 x 1024], 9 / 24 rows: 10.3 -> 8.2 / 15.1 ->
        // 11.8; eight waves 9.9 / 13.9).  12 waves with one tile row and 16 rows of x in the formats of four bits, where the walk's latency counts
        // more than what each wave adds of the sums and of x, of which there is less with fewer rows (rows past M are read as the last one).
        // 12 against 8 at 9 / 11 / 13 / 16 rows, averages over 19 weights of 512 to 4096 rows: row-major sym_int4 0.97 / 0.97 / 0.98 /
        // 0.99, asym_int4 0.94 / 0.95 / 0.95 / 0.97; tiled, 13 to 29 groups, 0.98 / 1.00 / 1.02 / 1.03 and 0.98 / 0.99 / 1.00 / 1.02; 12
        // groups, one round of waves, 1.01 / 0.98 / 0.98 / 0.97 and 1.01 / 0.99 / 1.00 / 1.00; 30 and more 0.94 / 0.97 / 0.99 / 1.01 and 0.96 /
        // 0.97 / 0.98 / 1.00, 1.03 at worst from 13 rows on.  nf4, tiled, 0.97 / 0.98 / 0.98 / 0.99 over all of them (row-major 0.99 / 0.99 / 1.00 /
        // 1.00); sym_int8 0.98 at 9 rows and up to 1.06 at 16, fp8_e4m3 0.98 and up to 1.08 from 12 on.
        if (M > 32 || (M <= 8 && !shared_by_three)) return none;
        if (rounds == 1 && MB == 1) {
            const bool int4 = qtype == QT_SYM_INT4 || qtype == QT_ASYM_INT4, tiled = layout == LAYOUT_TILED;
            const int most = int4 ? (tiled && G > 12 && G < 30 ? 10 : 13) : qtype == QT_NF4 && tiled ? 16 : 0;      // rows of x
            return {1, M <= most ? 12 : 8};
        }
        if (rounds <= 3) return {rounds, 8};
        if (rounds == 4) return layout == LAYOUT_TILED && MB == 1 ? WideShape{4, 8} : WideShape{2, 4};
        return {3, 4};
    }
    if (M > 64) return none;
    if (layout == LAYOUT_GGML) {
        // From 5 rows on: the streaming kernel reads unaligned weights in smaller pieces ([8008 x 8256], sym_int4, 8 rows:
        // 19.4 -> 15.2 us; 16 rows of [4001 x 2112] 7.1 -> 4.6).  Not fp8_e4m3, whose rows are whole and aligned, up to 16 rows.  17 .. 64 rows: against the row-major GEMM, whose 64-column tiles leave most
        // CUs idle at that size ([4001 x 2112], 24 / 64 rows: 11.4 -> 5.8 / 14.8 -> 8.6 us).
        const bool int4 = qtype == QT_SYM_INT4 || qtype == QT_ASYM_INT4;
        if (MB == 1) {
            // Beyond 1024 tile rows 9 .. 16 rows and 24 groups or more (9 / 16 rows on [17001 x 4096] 0.72 .. 0.85 / 0.75 .. 0.85 of
            // the streaming kernel's time over the formats, on [50001 x 4096] 0.81 .. 0.95 / 0.81 .. 0.98, on [17001 x 1024] 0.88 ..
            // 1.05); between 1537 and 2048, where that kernel's rounds come out even, four waves with four tile rows, and not fp8_e4m3
            // (1.03), nor asym_int4 up to 12 rows (9 / 16 rows on [32003 x 4096] 1.04 / 0.88; sym_int4 0.97 / 0.92).
            if (linear && T > 1024 && M > 8 && G >= 24) {
                if (T <= 1536 || T > 2048) return {2, 8};
                if (qtype != QT_FP8_E4M3 && (qtype != QT_ASYM_INT4 || M > 12)) return {4, 4};
            }
            if (M <= 4 || T > 1024 || qtype == QT_FP8_E4M3) return none;
            if (rounds == 1) return {1, 12};
            return {rounds == 3 && !int4 ? 1 : rounds, 8};                  // (more registers per tile: a third of them waits)
        }
        if (MB * G > 200 || (MB == 4 && T > 512) || (T > 1024 && (MB > 2 || qtype == QT_SYM_INT8))) return none;
    } else {
        // Up to 16 rows and beyond 1024 tile rows: workgroups of four waves, two to a CU, and as many tile rows as let 512 of them cover
        // the weight, in several rounds three.  9 and 16 rows, over the formats and types: 0.74 .. 0.96 of the streaming kernel's time on
        // 17008 .. 24576 weight rows (sym_int4 on [22016 x 4096] 17.6 -> 14.2 us), 0.86 .. 1.0 on [28672 x 4096] (level with 8 groups, not
        // taken), 0.85 .. 0.95 on 36000 rows.  5 .. 8 rows: asym_int4 and sym_int8, whose unpacking is what the streaming kernel spends its time
        // on there (0.86 .. 0.92 on [20480 x 4096] and [24576 x 4096], 1.0 .. 1.08 on [17008 x 4096]; the other formats 0.97 .. 1.06).
        const WideShape many = T <= 1536 || T > 2048 ? WideShape{3, 4} : WideShape{4, 4};
        if (M <= 8) {
            if (shared_by_three) return {3, 8};
            // two tile rows from 64 groups on (8 rows on [5008 x 11008] 0.86 .. 0.94; just above 256 tile rows half of the CUs would
            // have nothing, 6 rows on [4272 x 8192] in fp8_e4m3 1.08), 512 of them in the 8-bit formats only (0.91 .. 0.93,
            // the others 0.99 .. 1.04)
            const bool eight_bit = qtype == QT_SYM_INT8 || qtype == QT_FP8_E4M3;
            if (linear && M > 4 && rounds == 2 && T >= 304 && G >= 64 && (T < 512 || eight_bit)) return {2, 8};
            if (linear && M > 4 && T >= 1216 && G >= 24 && (qtype == QT_ASYM_INT4 || qtype == QT_SYM_INT8)) return many;
            return none;
        }
        if (MB == 1 && T > 1024) return !linear || (T > 1536 && T <= 2048 && G < 24) ? none : many;
        if ((MB > 1 && MB * G > 192) || (MB == 4 && T > 768) || (T > 1024 && MB > 2)) return none;
    }
    if (T > 1024) return {4, 4};
    return {rounds, MB == 1 && rounds == 1 ? 12 : 8};
}

static int format_index(int qtype) {
    return qtype == QT_SYM_INT4 ? 0 : qtype == QT_ASYM_INT4 ? 1 : qtype == QT_SYM_INT8 ? 2 : qtype == QT_NF4 ? 3 : 4;
}

// What a launch takes whose workgroups are one per CU at most, 8 waves each, with r tile rows and 16 * mb rows of x to a workgroup:
// microseconds, fitted to 1250 sizes (M = 17 .. 900, N to 16384, K to 14000) in up to three shapes each, 6 to 10 % rms.  A launch; per
// 1024 columns what goes with the groups, with x, with the weights and with their products; the sums; x out of L2.  x's type counts in row-major
// nf4 only, three operands in bfloat16 and two in fp16, and is left out: 1.02 .. 1.08 of the fp16 time with up to six products (1.15 with eight and
// nine) where the row-major GEMM, which it is compared with, takes 1.11.
static double wide_us(int qtype, int layout, int r, int mb, int M, int T, int G) {
    static const double fit[2][5][7] = {                    // row-major, tiled; sym_int4, asym_int4, sym_int8, nf4, fp8_e4m3
        {{2.680, 0.076, 0.200, 0.466, 0.032, 0.249, 0.020}, {2.423, 0.326, 0.100, 0.390, 0.114, 0.296, 0.042},
         {2.388, 0.297, 0.040, 0.653, 0.088, 0.299, 0.036}, {3.236, 0.000, 0.000, 0.814, 0.158, 0.110, 0.057},
         {2.751, 0.133, 0.065, 0.365, 0.125, 0.135, 0.028}},
        {{2.975, 0.190, 0.075, 0.163, 0.126, 0.127, 0.038}, {3.089, 0.058, 0.118, 0.221, 0.132, 0.078, 0.038},
         {2.974, 0.087, 0.177, 0.415, 0.074, 0.094, 0.031}, {2.817, 0.170, 0.081, 0.279, 0.061, 0.160, 0.043},
         {3.052, 0.223, 0.102, 0.288, 0.096, 0.065, 0.034}}};
    const double(&f)[7] = fit[layout == LAYOUT_TILED][format_index(qtype)];
    const double wgs = (double)((T + r - 1) / r) * ((M + 16 * mb - 1) / (16 * mb));
    return f[0] + (G + 7) / 8 * (f[1] + f[2] * mb + f[3] * r + f[4] * r * mb) + f[5] * r * mb + f[6] * wgs / 256 * G * mb;
}

// Rows of x dealt to several workgroups: so many rows and tile rows to each that the workgroups are one per CU at most and the estimate is
// the shortest; r = 0: there is no such shape.  r * mb products of 16 x 16: up to nine, six in asym_int4, is what the estimates were fitted to.
// (No form of these spills, from twelve on all but fp8_e4m3 do, but for four tile rows and two blocks of row-major nf4 in bfloat16, whose weights are
// three operands: six registers, in the loop.  146 to 160 rows on 3100 .. 3250 weight rows, that form against the row-major GEMM: 0.66 .. 0.88 of
// its time up to 1344 columns, 0.98 .. 1.03 at 1600 .. 1920, 0.92 .. 0.96 at 2112 .. 2432, 1.01 .. 1.07 at 2816 .. 3904: up to 20 groups.)
static WideShape wide_batch_shape(int qtype, int layout, int dt, int M, int N, int K, double *us) {
    WideShape best = {0, 0};
    if (M <= 16 || M > 1024 || K > 16384) return best;
    const int T = (N + TILE_ROWS - 1) / TILE_ROWS, G = (K + TILE_COLS - 1) / TILE_COLS;
    for (int r = 1; r <= 4; r++)
        for (int mb = 1; mb <= 4 && r * mb <= (qtype == QT_ASYM_INT4 ? 6 : 9); mb++) {
            if ((int64_t)((T + r - 1) / r) * ((M + 16 * mb - 1) / (16 * mb)) > 256) continue;
            if (r == 4 && mb == 2 && layout == LAYOUT_GGML && qtype == QT_NF4 && dt == DT_BF16 && G > 20) continue;
            const double t = wide_us(qtype, layout, r, mb, M, T, G);
            if (!best.r || t < *us) {
                best = {r, 8, mb};
                *us = t;
            }
        }
    return best;
}

// Microseconds with rows dealt that way, 0 where there is no such shape: for the choice between this and the other kernels.  (What it takes
// the place of there: the K splits, half tiles and narrow tiles of the GEMMs, whose few tiles leave CUs idle or walk K at the latency of a
// step, and their sums.  128 rows on [2048 x 2048] 15.2 -> 7.0 us, 72 on [4096 x 4096] 19.3 -> 12.4, 217 on [1001 x 1024] row-major
// 11.3 -> 6.2, averages of the formats.)
double gemv_wide_batch_us(int qtype, int layout, int dt, int M, int N, int K) {
    double us = 0.0;
    return wide_batch_shape(qtype, layout, dt, M, N, K, &us).r ? us : 0.0;
}

// linear: also the sizes that wide_shape leaves to other kernels; r = 0: not a size for this kernel
WideShape gemv_wide_shape(int qtype, int layout, int dt, int M, int N, int K, bool linear) {
    const WideShape s = wide_shape(qtype, layout, dt, M, N, K, linear);
    const int T = (N + TILE_ROWS - 1) / TILE_ROWS, MB = (M + 15) / 16;
    if (dt == DT_F32) {
        // Up to 64 rows: 16 to a workgroup where the workgroups are then one per CU at most, with up to three tile rows (four in place of
        // two passes: 33 rows and more).  Two blocks of x take a workgroup longer than three tile rows.  Against wide_shape's shape, or two
        // passes, 170 random sizes of 17 .. 64 rows (N to 16384, K to 16384): 117 change, 0.78 of the time, four of them 1.02 .. 1.035 (20
        // rows on row-major [4141 x 5632] in fp8_e4m3 18.8 -> 19.2 us; 23 on [2032 x 4224] in sym_int4 14.0 -> 10.5, 51 on [1632 x 11008] 46.3 -> 23.3).
        for (int r = 1; MB > 1 && MB <= 4 && r <= (MB > 2 && layout == LAYOUT_TILED ? 4 : 3); r++)
            if ((T + r - 1) / r * MB <= 256) return {r, 8, 1};
        return s;
    }
    if (M <= 16 || (M > 64 && !linear) || (s.r && T > 1024)) return s;
    // 17 .. 64 rows, where the estimate is 5 % shorter; beyond 32 groups 8 % where a workgroup then has two tile rows more (35 rows on
    // [3584 x 6784] in nf4, three in place of one, estimated 7.8 % shorter, took 1.06 of the time), beyond 64 groups 12 % (18 rows on [5104 x
    // 9728] in asym_int4, estimated 8 % shorter, took 1.06).  453 of 698 random sizes, other ones than those of the fit, in 0.83 of the
    // time, 1.01 at worst
    const int G = (K + TILE_COLS - 1) / TILE_COLS;
    double us = 0.0;
    const WideShape dealt = wide_batch_shape(qtype, layout, dt, M, N, K, &us);
    if (!s.r) return linear ? dealt : s;
    return dealt.r && us < (G > 64 ? 0.88 : G > 32 && dealt.r > s.r + 1 ? 0.92 : 0.95) * wide_us(qtype, layout, s.r, MB, M, T, G) ? dealt : s;
}

// The fused gate/up form: R of either weight, so at most 2.  Against two launches' worth of streaming passes and the fused
// form of the tiled GEMM, which has few tiles at these sizes and walks all of K in each (fp16 sym_int4 [11008 x 4096] at 12 /
// 24 / 48 rows 18.0 -> 14.2 / 31.1 -> 19.9 / 40.9 -> 28.8 us, [4096 x 16384] at 24 rows 127 -> 26).
static WideShape wide_mlp_shape(int qtype, int act_dtype, int M, int N, int K) {
    const int T = N / TILE_ROWS, MB = (M + 15) / 16, rounds = (T + 255) / 256;
    const WideShape none = {0, 0};
    // 5 .. 8 rows: where the streaming kernel spends more on unpacking than on memory
    if (M <= 8 && !(M > 4 && (qtype == QT_SYM_INT8 || (qtype == QT_NF4 && T >= 512)))) return none;
    if (M > 64 || (MB > 2 && T > 1024)) return none;
    // One tile row of either weight where that takes an odd number of rounds, with 16 rows and the formats of many registers,
    // and with 49 .. 64 rows where two spill.  8 waves where a CU has one workgroup, else 4.
    const bool small = qtype == QT_SYM_INT4 || qtype == QT_NF4;
    const int r = rounds == 1 || rounds == 3 || (MB == 1 && !small) || !wide_mlp_two_rows(qtype, act_dtype == DT_F16, MB) ? 1 : 2;
    return {r, (T + r - 1) / r <= 256 ? 8 : 4};
}

// The fused form with rows of x dealt to several workgroups, as wide_batch_shape, r of either weight; r = 0: no such shape, or the fused
// form of the tiled GEMM is the faster one.  Fitted to 920 launches (M = 17 .. 600, N to 16384, K to 14000), 7 to 8 % rms.  17 .. 64 rows: ahead
// of the shape with all rows to a workgroup where the estimate is shorter, beyond 8 groups 3 % shorter (34 rows on [2368 x 2048] in fp8_e4m3, estimated 2 % shorter,
// took 1.10).  216 of 330 random sizes, other ones than those of the fit, in 0.83 of the time.  More: against narrow tiles, which
// while they are one per CU take 4 to 5 us and 0.54 to 0.65 per 128 columns (118 of 147 random sizes 0.61 of the time, none longer).
static WideShape wide_mlp_batch_shape(int qtype, int act_dtype, int M, int N, int K) {
    static const double fit[5][7] = {{3.495, 0.036, 0.213, 0.220, 0.080, 0.044, 0.030}, {3.097, 0.004, 0.097, 0.235, 0.141, 0.139, 0.041},
                                     {3.434, 0.091, 0.134, 0.416, 0.039, 0.063, 0.043}, {3.493, 0.000, 0.116, 0.322, 0.085, 0.088, 0.031},
                                     {3.293, 0.115, 0.195, 0.351, 0.018, 0.054, 0.043}};
    static const double tiled[5][2] = {{4.36, 0.579}, {4.32, 0.537}, {4.05, 0.580}, {4.84, 0.648}, {4.20, 0.545}};
    WideShape best = {0, 0};
    if (M <= 16 || M > 1024 || K > 16384) return best;
    const int T = N / TILE_ROWS, G = K / TILE_COLS, q = format_index(qtype);
    const double(&f)[7] = fit[q];
    auto workgroups = [&](int r, int mb) { return (int64_t)((T + r - 1) / r) * ((M + 16 * mb - 1) / (16 * mb)); };
    auto estimate = [&](int r, int mb) {
        return f[0] + (G + 7) / 8 * (f[1] + f[2] * mb + f[3] * 2 * r + f[4] * 2 * r * mb) + f[5] * 2 * r * mb
            + f[6] * (double)workgroups(r, mb) / 256 * G * mb;
    };
    double us = M <= 64 ? 1e30 : 0.95 * (tiled[q][0] + tiled[q][1] * G);
    for (int r = 1; r <= 2; r++)
        for (int mb = 1; r * mb <= 4; mb++) {
            if (workgroups(r, mb) > 256) continue;
            const double t = estimate(r, mb);
            if (t < us) {
                best = {r, 8, mb};
                us = t;
            }
        }
    const WideShape all = wide_mlp_shape(qtype, act_dtype, M, N, K);
    const int MB = (M + 15) / 16;
    return best.r && all.r && workgroups(all.r, MB) <= 256 && us >= (G > 8 ? 0.97 : 1.0) * estimate(all.r, MB) ? all : best;
}

bool gemv_wide_applies(int qtype, int layout, int act_dtype, int M, int N, int K) {
    return wide_shape(qtype, layout, act_dtype, M, N, K, true).r != 0;
}

// s: from gemv_wide_shape
int launch_gemv_wide(const void *x, const void *w, const void *bias, void *y, int qtype, int layout, int act_dtype, int M, int N, int K,
                     const WideShape &s, hipStream_t st) {
    switch (qtype) {
    case QT_SYM_INT4: return launch_wide_q<QT_SYM_INT4>(x, w, bias, y, layout, act_dtype, M, N, K, s, st);
    case QT_ASYM_INT4: return launch_wide_q<QT_ASYM_INT4>(x, w, bias, y, layout, act_dtype, M, N, K, s, st);
    case QT_SYM_INT8: return launch_wide_q<QT_SYM_INT8>(x, w, bias, y, layout, act_dtype, M, N, K, s, st);
    case QT_NF4: return launch_wide_q<QT_NF4>(x, w, bias, y, layout, act_dtype, M, N, K, s, st);
    case QT_FP8_E4M3: return launch_wide_q<QT_FP8_E4M3>(x, w, bias, y, layout, act_dtype, M, N, K, s, st);
    default: return -2;
    }
}

// linear: also above 64 rows, on small weights; r = 0: not a size for this kernel
WideShape mlp_wide_shape(int qtype, int act_dtype, int M, int N, int K, bool linear) {
    WideShape s = {0, 0};
    if (M <= 64 || linear) s = wide_mlp_batch_shape(qtype, act_dtype, M, N, K);
    return s.r ? s : wide_mlp_shape(qtype, act_dtype, M, N, K);
}

// s: from mlp_wide_shape
int launch_mlp_wide(const void *x, const void *wg, const void *wu, void *y, int qtype, int act_dtype, int M, int N, int K, int act,
                    const WideShape &s, hipStream_t st) {
    switch (qtype) {
    case QT_SYM_INT4: return launch_wide_mlp_q<QT_SYM_INT4>(x, wg, wu, y, act_dtype, M, N, K, act, s, st);
    case QT_ASYM_INT4: return launch_wide_mlp_q<QT_ASYM_INT4>(x, wg, wu, y, act_dtype, M, N, K, act, s, st);
    case QT_SYM_INT8: return launch_wide_mlp_q<QT_SYM_INT8>(x, wg, wu, y, act_dtype, M, N, K, act, s, st);
    case QT_NF4: return launch_wide_mlp_q<QT_NF4>(x, wg, wu, y, act_dtype, M, N, K, act, s, st);
    case QT_FP8_E4M3: return launch_wide_mlp_q<QT_FP8_E4M3>(x, wg, wu, y, act_dtype, M, N, K, act, s, st);
    default: return -2;
    }
}

}  // namespace lowbit
