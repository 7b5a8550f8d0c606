// One pass over the weights for up to 64 rows of x (serving batches): y[M,N] = x[M,K] * dequant(W)[N,K]^T.  More rows, where the
// weight is small: so many rows to a workgroup, that the workgroups are one per CU (gemv_wide.hip).
//
// A workgroup owns R tile rows (16 weight rows each) for all of K; its waves take the 128-column groups of K in turn.
// Each wave copies its group of x (16 * MB rows) into a private part of LDS and multiplies it with R weight tiles, whose
// registers already are the MFMA operand: exact codes, the block scale applied to the fp32 results, as in the streaming
// kernel for up to 16 rows (gemv.hip).  The loads of a wave's next group go out before the current one is computed - x
// into the registers that its LDS copy has freed, the weights into a second set - so that a walk of a few groups costs
// one memory latency and not one per group.  The waves' partial sums meet in LDS: no workspace, no second launch.
//
// What bounds it: every workgroup reads all of x from L2 (40 rows of 4096: 327 KB, against 36 KB of sym_int4 weights per
// tile row), which is why R tile rows share it, and the scale: MB * 4 FMAs per 8 codes and lane next to some nine
// instructions of unpacking.  Measured against the kernels it takes the place of (ring and its reduction, K splits of the
// tiled GEMM, two and three passes of the streaming kernel), each launch on weights it has not just read, sym_int4 fp16:
// [12288 x 4096] at 9 / 24 / 32 / 48 / 64 rows 10.5 -> 8.4 / 15.1 -> 11.2 / 15.7 -> 11.5 / 19.0 -> 15.7 / 20.5 -> 17.9 us,
// [4096 x 4096] at 24 / 48 rows 10.5 -> 7.3 / 14.6 -> 9.7, [5632 x 2048] at 32 rows 11.6 -> 6.1; over 504 points (seven
// shapes and more, five formats, 9 .. 64 rows) the best shape of this kernel is 1.26 times faster on average.
//
// This header holds the kernel and the launch code of one weight format; gemv_wide_<format>.hip instantiate it,
// gemv_wide.hip decides where it is used.
#pragma once
#include "lowbit_rows.h"
#include "lowbit_unpack.h"
#include "lowbit_wide_plan.h"

#include <type_traits>

namespace lowbit {

// F32: x, bias and y are float, x as two bf16 planes (see gemv.hip).  ROWS: row-major weights of any shape
// (lowbit_rows.h).  DUAL: the fused gate/up projection, act(x Wg^T) * (x Wu^T): R tile rows of either weight.
// wide_max_waves: what gemv_wide.hip asks for at most, and with it the registers a wave may have (256 at 8, 168 at
// 12).  Four tiles in the 128 that 16 waves leave spilled: 16 rows on [14336 x 4096], asym_int4 bf16 20.6 ->
// 12.7 us, sym_int8 23.3 -> 16.0.
constexpr int wide_max_waves(int mb, int tiles) { return mb == 1 && tiles == 1 ? 12 : 8; }

// 16-byte chunks from the first of four 16-bit rows of x to row xrow (0 .. 3) of them, or to the last row where fewer than xrow are
// left; K is a multiple of 128.  (In elements three rows are past 32 bits from K = 1.4 * 10^9 on; a 64-bit offset costs 0.5 %
// on average over 700 points, 6 % at worst.)
__host__ __device__ inline uint32_t wide_row_chunks(int xrow, int left, int K) {
    const uint32_t row = (uint32_t)K / 8u, at = (uint32_t)xrow * row, most = (uint32_t)(left < 3 ? left : 3) * row;
    return at < most ? at : most;
}

// Whether a form's last group stands apart (PEEL in the kernel)
template <int QT, typename AT, int MB, int R, bool F32, bool ROWS, bool DUAL> constexpr bool wide_peels() {
    return !ROWS && !F32 && (DUAL ? 2 * R : R) * MB <= (QT == QT_ASYM_INT4 ? 6 : QT == QT_SYM_INT8 || Operand<QT, AT, F32, ROWS>::NEED_S ? 8 : 9);
}

// CROWD: the fused form without PEEL, see launch_wide_r
template <int QT, typename AT, int MB, int R, bool F32, bool ROWS, bool DUAL, bool CROWD = false>
__global__ __launch_bounds__(64 * wide_max_waves(MB, DUAL ? 2 * R : R)) void gemv_wide_kernel(
    const void *__restrict__ x_, const uint8_t *__restrict__ w, const uint8_t *__restrict__ w_up, const void *__restrict__ bias_,
    void *__restrict__ y_, int M, int N, int K, int act) {
    using F = Fmt<QT>;
    using V8 = typename Vec8<AT>::type;
    using ET = typename std::conditional<F32, float, AT>::type;
    using Op = Operand<QT, AT, F32, ROWS>;
    constexpr float OFFSET = Op::OFFSET;
    constexpr bool NEED_S = Op::NEED_S;
    constexpr int PARTS = Op::PARTS;
    // Steps of 32 columns per scale.  PEEL: the MFMAs of a block follow each other into one result, which is scaled once (nf4: half as
    // many FMAs, fp8_e4m3: a quarter; 40 rows on [11008 x 4096] in nf4 16.4 -> 15.5 us, in fp8_e4m3 16.7 -> 16.2, 24 on [5200 x 9728] in
    // nf4 17.6 -> 16.9; 0.985 of the time over 56 sizes, formats and types, none longer by more than the runs differ).
    constexpr int SUB = F::QK / 32;
    static_assert(SUB == 1 || !NEED_S, "the row sums of x are taken step by step");
    constexpr int NT = DUAL ? 2 * R : R;                     // weight tiles per group; DUAL: R of the gate, R of the up weight
    // PEEL: a wave's last group, which loads nothing, stands apart from the loop, and the order of the products is given.  With a
    // condition around the loads the compiler merged the registers of two groups' weights where the ways met, in the middle of the
    // products, and waited there for the loads that it had just issued; and it let most products wait for their MFMA.  It takes
    // some 40 registers more, so only where they are there: with spills a kernel took up to 1.6 times as long.  Old / new
    // form, fp16 sym_int4: 40 rows on [11008 x 4096] 16.3 / 14.7 us, on [6144 x 2048] 8.6 / 7.7, 64 on [4096 x 4096] 13.7 / 12.2,
    // 12 on [11008 x 4096] 9.4 / 8.7; 1.05 on average.  Row-major weights and float32 activations: level, not taken.
    constexpr bool PEEL = !CROWD && wide_peels<QT, AT, MB, R, F32, ROWS, DUAL>();
    static_assert(!DUAL || (!F32 && !ROWS), "the fused form takes 16-bit activations and tiled weights");
    constexpr int PLANE = 16 * MB * 256, XBYTES = PLANE * (F32 ? 2 : 1), XC = 4 * MB;     // bytes of x in LDS; chunks of 8 per lane
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    // (one wait for all arguments and the number of threads: left alone the compiler loaded that one behind the others, a scalar load's time
    // that 40 rows on [11008 x 4096] took 13.4 -> 14.0 us for)
    const int threads = (int)blockDim.x;
    asm volatile("" :: "s"(x_), "s"(w), "s"(M), "s"(N), "s"(K), "s"(threads));
    // (blockIdx.y: which 16 * MB rows of x)
    const int m0 = (int)blockIdx.y * 16 * MB;
    const ET *const x = (const ET *)x_ + (int64_t)m0 * K;
    ET *const y = (ET *)y_ + (int64_t)m0 * N;
    M = M - m0 < 16 * MB ? M - m0 : 16 * MB;
    const int lane = threadIdx.x & 63, W = threads >> 6, r = lane & 15, c = lane >> 4;
    const int wave = PEEL ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : threadIdx.x >> 6;
    uint8_t *const xs = smem + wave * XBYTES;
    const int G = ROWS ? (K + TILE_COLS - 1) / TILE_COLS : K / TILE_COLS, blocks = K / F::QK;

    gbytes wr[NT];                                           // ROWS: this lane's weight row; tiled: the tile row
#pragma unroll
    for (int wi = 0; wi < NT; wi++) {
        const int64_t row = (int64_t)blockIdx.x * R + wi % R;
        if constexpr (ROWS) {
            const int64_t n = row * TILE_ROWS + r;
            wr[wi] = (gbytes)w + (n < N ? n : N - 1) * (int64_t)blocks * F::TS;
        } else {
            const int64_t last = N / TILE_ROWS - 1;          // (tile rows past N are computed and not stored)
            wr[wi] = (gbytes)(wi < R ? w : w_up) + (row < last ? row : last) * (int64_t)G * F::TILE_BYTES;
        }
    }
    // x: 16 consecutive lanes load the 16 chunks of a row's group (256 bytes; F32: 512), four rows per instruction
    const int u = lane & 15, xrow = lane >> 4;
    auto load = [&](int g, u32x4 (&xv)[F32 ? 2 * XC : XC], auto &t, bool first_group = false) __attribute__((always_inline)) {
        const int col = g * TILE_COLS + u * 8;
        const bool past = ROWS && col >= K;                  // (put makes zeros of columns past K)
#pragma unroll
        for (int i = 0; i < XC; i++) {
            const u32x4 *p;
            if constexpr (PEEL) {                            // a scalar base per instruction, one lane offset
                const int first = 4 * i < M ? 4 * i : (M - 1) & ~3;
                p = (const u32x4 *)(x + (int64_t)first * K + g * TILE_COLS) + (wide_row_chunks(xrow, M - 1 - first, K) + (uint32_t)u);
            } else {
                const int m = i * 4 + xrow;
                p = (const u32x4 *)(x + (int64_t)(m < M ? m : M - 1) * K + (past ? K - 8 : col));
            }
#pragma unroll
            for (int h = 0; h < (F32 ? 2 : 1); h++) xv[i * (F32 ? 2 : 1) + h] = p[h];
            // (ahead of the loop each goes out as its address is there: left alone the compiler kept all of them behind the last one's)
            if (first_group) __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int wi = 0; wi < NT; wi++) {
            if constexpr (ROWS) load_rows<QT>(wr[wi], g, c, blocks, t[wi]);
            else load_tile<QT, true>(wr[wi] + (int64_t)g * F::TILE_BYTES, lane, r, t[wi]);
        }
    };
    // Unit v (16 bytes) of row m lies at unit v ^ m % 16: the rows are 256 bytes apart, and a step reads one unit of 16 of
    // them at a time.
    auto put = [&](int g, const u32x4 (&xv)[F32 ? 2 * XC : XC]) __attribute__((always_inline)) {
        // (here and not where they are loaded: there the select would wait for the loads, in front of the previous group)
        const bool past = ROWS && g * TILE_COLS + u * 8 >= K;
        const u32x4 none = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int i = 0; i < XC; i++) {
            const int m = i * 4 + xrow;
            auto one = [&](uint8_t *row, const u32x4 &v) __attribute__((always_inline)) {
                if constexpr (ROWS) store_x_rows<QT>(row, u, v, m & 15);
                else *(u32x4 *)(row + (u ^ (m & 15)) * 16) = v;
            };
            if constexpr (F32) {
                u32x4 hi, lo;
                split_f32<false>(past ? none : xv[2 * i], past ? none : xv[2 * i + 1], hi, lo);
                one(xs + m * 256, hi);
                one(xs + PLANE + m * 256, lo);
            } else {
                one(xs + m * 256, past ? none : xv[i]);
            }
        }
    };

    f32x4 acc[NT][MB];
#pragma unroll
    for (int wi = 0; wi < NT; wi++)
#pragma unroll
        for (int mb = 0; mb < MB; mb++) acc[wi][mb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    const f32x4 zero4 = {0.0f, 0.0f, 0.0f, 0.0f};
    const V8 ones = ones8<AT>();
    const Op op;

    typename std::conditional<ROWS, RowRegs<QT>, TileRegs<QT>>::type wc[NT], wn[NT];
    u32x4 xv[F32 ? 2 * XC : XC];
    if constexpr (PEEL) {
        load(wave, xv, wn, true);                            // (no more waves than groups)
        auto hold = [](auto &t) __attribute__((always_inline)) {
            asm volatile("" : "+v"(t.q0));
            if constexpr (F::BITS == 8) asm volatile("" : "+v"(t.q1));
        };
        auto group = [&](int g, auto more_) __attribute__((always_inline)) {
            constexpr bool more = decltype(more_)::value;
#pragma unroll
            for (int wi = 0; wi < NT; wi++) {
                wc[wi] = wn[wi];
                hold(wc[wi]);
            }
            // the LDS part is private to the wave, whose LDS operations execute in order: a fence for the compiler is enough
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            put(g, xv);
            if constexpr (more) load(g + W, xv, wn);
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            // Unit q = (step j, 16-row block mb), in the order the hardware should issue them: the MFMAs of a unit, the LDS read of
            // the next one's x, the scaling of the unit before, whose results have landed meanwhile.
            auto read_x = [&](int q) __attribute__((always_inline)) {
                return *(const V8 *)(xs + (q % MB * 16 + r) * 256 + (((q / MB * 4 + c) ^ r) * 16));
            };
            V8 a[2], b[NT][PARTS];
            float d[2][NT], e[2][NT];                             // of this block and the one before
            f32x4 run[NT][MB], p[2][NT], s[2];                    // a block's products so far; those of whole blocks
            a[0] = read_x(0);
#pragma unroll
            for (int q = 0; q <= 4 * MB; q++) {
                if (q < 4 * MB) {
                    const int j = q / MB;
                    if (q % MB == 0) {
#pragma unroll
                        for (int wi = 0; wi < NT; wi++) {
#pragma unroll
                            for (int part = 0; part < PARTS; part++) b[wi][part] = op.get(wc[wi], j, part);
                            if (j % SUB) continue;
                            const int k = j / SUB & 1;
                            float mn;
                            tile_scale<QT>(wc[wi], j, d[k][wi], mn);
                            e[k][wi] = mn - OFFSET * d[k][wi];
                            d[k][wi] = Op::scale(d[k][wi]);
                        }
                    }
                    s[q & 1] = NEED_S ? mfma16(a[q & 1], ones, zero4) : zero4;
#pragma unroll
                    for (int wi = 0; wi < NT; wi++) {
                        f32x4 &sum = run[wi][q % MB];
                        sum = Op::product(a[q & 1], a[q & 1], b[wi], j % SUB ? sum : zero4);
                        p[q & 1][wi] = sum;
                    }
                    if (q + 1 < 4 * MB) a[(q + 1) & 1] = read_x(q + 1);
                }
                if (q > 0 && ((q - 1) / MB + 1) % SUB == 0) {
                    const int o = (q - 1) & 1, mb = (q - 1) % MB, k = (q - 1) / MB / SUB & 1;
#pragma unroll
                    for (int wi = 0; wi < NT; wi++)
#pragma unroll
                        for (int i = 0; i < 4; i++)
                            acc[wi][mb][i] = Op::add(acc[wi][mb][i], d[k][wi], p[o][wi][i], e[k][wi], s[o][i]);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        int g = wave;
        for (; g + W < G; g += W) group(g, std::true_type{});
        group(g, std::false_type{});
    } else {
        const int first = wave < G ? wave : G - 1;
        load(first, xv, wn);
        for (int g = wave; g < G; g += W) {
#pragma unroll
            for (int wi = 0; wi < NT; wi++) wc[wi] = wn[wi];
            // the LDS part is private to the wave, whose LDS operations execute in order: a fence for the compiler is enough
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            put(g, xv);
            if (g + W < G) load(g + W, xv, wn);
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            uint32_t hb[NT][4];
            if constexpr (ROWS) {
#pragma unroll
                for (int wi = 0; wi < NT; wi++) arrange_rows<QT>(wc[wi], hb[wi]);
            }
#pragma unroll
            for (int j = 0; j < 4; j++) {
                V8 b[NT][PARTS];
                float d[NT], e[NT];
#pragma unroll
                for (int wi = 0; wi < NT; wi++) {
#pragma unroll
                    for (int part = 0; part < PARTS; part++) b[wi][part] = op.get(wc[wi], j, part);
                    float mn;
                    if constexpr (ROWS) hdr_to_scale<QT>(hb[wi][j], d[wi], mn);
                    else tile_scale<QT>(wc[wi], j, d[wi], mn);
                    e[wi] = mn - OFFSET * d[wi];
                    d[wi] = Op::scale(d[wi]);
                }
#pragma unroll
                for (int mb = 0; mb < MB; mb++) {
                    const uint8_t *at = xs + (mb * 16 + r) * 256 + (((j * 4 + c) ^ r) * 16);
                    const V8 a = *(const V8 *)at;
                    V8 al;
                    if constexpr (F32) al = *(const V8 *)(at + PLANE);
                    f32x4 s = zero4;
                    if constexpr (NEED_S) {
                        s = mfma16(a, ones, zero4);
                        if constexpr (F32) s = mfma16(al, ones, s);
                    }
#pragma unroll
                    for (int wi = 0; wi < NT; wi++) {
                        const f32x4 p = Op::product(a, al, b[wi]);
#pragma unroll
                        for (int i = 0; i < 4; i++) acc[wi][mb][i] = Op::add(acc[wi][mb][i], d[wi], p[i], e[wi], s[i]);
                    }
                }
#pragma unroll
                for (int wi = 0; wi < NT; wi++)                   // one step after the other: the scheduler would gather all reads first
#pragma unroll
                    for (int mb = 0; mb < MB; mb++) asm volatile("" : "+v"(acc[wi][mb]));
            }
        }
    }

    // The waves' sums meet in their parts of LDS; C layout: lane = 16*grp + weight row, register i = row 4*grp + i of x.
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    constexpr int RS = XBYTES / 16;                          // f32x4 per wave's part: at least NT * MB * 64
    static_assert(NT * MB * 1024 <= XBYTES, "partial sums fit the x part");
    f32x4 *const red = (f32x4 *)smem;
#pragma unroll
    for (int wi = 0; wi < NT; wi++)
#pragma unroll
        for (int mb = 0; mb < MB; mb++) red[wave * RS + (wi * MB + mb) * 64 + lane] = acc[wi][mb];
    __syncthreads();
    for (int q = wave; q < R * MB; q += W) {
        const int wi = q / MB, mb = q % MB;
        f32x4 s = red[q * 64 + lane], up = zero4;
        for (int v = 1; v < W; v++) s += red[v * RS + q * 64 + lane];
        if constexpr (DUAL) {
            for (int v = 0; v < W; v++) up += red[v * RS + (R * MB + q) * 64 + lane];
        }
        const int64_t n = ((int64_t)blockIdx.x * R + wi) * TILE_ROWS + r;
        if (n >= N) continue;
        const float bv = bias_ ? (float)((const ET *)bias_)[n] : 0.0f;
        auto store = [&](int m, float s, float up) __attribute__((always_inline)) {
            const float v = DUAL ? gate_act(s, act) * up : s + bv;
            if constexpr (F32) y[(int64_t)m * N + n] = v;
            else y[(int64_t)m * N + n] = to_at<AT>(v);
        };
        uint32_t again = 0;                                   // results that are not finite, see dot_fp32
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int m = mb * 16 + c * 4 + i;
            if (m < M) {
                store(m, s[i], up[i]);
                again |= __builtin_isfinite(s[i]) && __builtin_isfinite(up[i]) ? 0u : 1u << i;
            }
        }
        for (; again; again &= again - 1) {
            const int m = mb * 16 + c * 4 + __builtin_ctz(again);
            const ET *row = x + (int64_t)m * K;
            store(m, dot_fp32<QT, ROWS>(row, w, n, K), DUAL ? dot_fp32<QT, ROWS>(row, w_up, n, K) : 0.0f);
        }
    }
}

// Workgroups of four waves that the GPU holds at once, in either form
struct WideRoom {
    int peel, crowd;
};
inline WideRoom wide_room(const void *peel, const void *crowd, size_t lds) {
    int dev = 0, cus = 0, a = 0, b = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&a, peel, 256, lds) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&b, crowd, 256, lds) != hipSuccess) return {0, 0};
    return {a * cus, b * cus};
}

template <int QT, typename AT, int MB, int R, bool F32, bool ROWS, bool DUAL>
static int launch_wide_r(const void *x, const void *w, const void *w_up, const void *bias, void *y, int M, int N, int K, int act,
                         int waves, hipStream_t st) {
    constexpr int XBYTES = 16 * MB * 256 * (F32 ? 2 : 1), LDS = 128 * 1024, MOST = wide_max_waves(MB, DUAL ? 2 * R : R);
    auto kern = gemv_wide_kernel<QT, AT, MB, R, F32, ROWS, DUAL>;
    const int G = (K + TILE_COLS - 1) / TILE_COLS;
    int wv = LDS / XBYTES;
    wv = wv > MOST ? MOST : wv;
    wv = wv > waves ? waves : wv;
    wv = wv > G ? G : wv;
    // the default limit of dynamic LDS is 64 KB; raised once per process (thread-safe static), on the one GPU this library drives
    static const hipError_t raised = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
    if (raised != hipSuccess) return -6;
    const int wgs = (N + TILE_ROWS * R - 1) / (TILE_ROWS * R);
    if constexpr (DUAL && wide_peels<QT, AT, MB, R, F32, ROWS, DUAL>()) {
        // The registers of PEEL let a CU hold fewer workgroups of four waves, in several of these forms two in place of three:
        // with more than that the others wait for a second round.  With PEEL / without: 22 rows on [9376 x 768] in bf16 sym_int4
        // 9.0 / 7.4 us, 37 on [10336 x 768] in fp16 nf4 11.0 / 9.8, 26 on [9920 x 1152] in bf16 sym_int8 12.3 / 10.5.
        auto crowd = gemv_wide_kernel<QT, AT, MB, R, F32, ROWS, DUAL, true>;
        static const WideRoom room = wide_room((const void *)kern, (const void *)crowd, 4 * XBYTES);
        if (wv == 4 && room.crowd > room.peel && wgs > room.peel) kern = crowd;
    }
    hipLaunchKernelGGL(kern, dim3(wgs, (M + 16 * MB - 1) / (16 * MB)), dim3(64 * wv), (size_t)wv * XBYTES, st, x, (const uint8_t *)w, (const uint8_t *)w_up, bias, y, M, N, K, act);
    return 0;
}

// -7: a shape that is not instantiated (the caller, gemv_wide.hip, asks for none)
template <int QT, typename AT, int MB, bool F32, bool ROWS>
static int launch_wide_mb(const void *x, const void *w, const void *bias, void *y, int M, int N, int K, const WideShape &s, hipStream_t st) {
    if (s.r == 1) return launch_wide_r<QT, AT, MB, 1, F32, ROWS, false>(x, w, nullptr, bias, y, M, N, K, 0, s.waves, st);
    if (s.r == 2) return launch_wide_r<QT, AT, MB, 2, F32, ROWS, false>(x, w, nullptr, bias, y, M, N, K, 0, s.waves, st);
    if (s.r == 3) return launch_wide_r<QT, AT, MB, 3, F32, ROWS, false>(x, w, nullptr, bias, y, M, N, K, 0, s.waves, st);
    if constexpr (!F32 || (MB == 1 && !ROWS)) {
        if constexpr (MB < 4)
            if (s.r == 4) return launch_wide_r<QT, AT, MB, 4, F32, ROWS, false>(x, w, nullptr, bias, y, M, N, K, 0, s.waves, st);
    }
    return -7;
}

template <int QT, typename AT, bool F32, bool ROWS>
static int launch_wide_t(const void *x, const void *w, const void *bias, void *y, int M, int N, int K, const WideShape &s, hipStream_t st) {
    const int mb = s.mb ? s.mb : (M + 15) / 16;
    if (M > 16 * mb * 65535) return -7;                      // (blocks of rows are counted in the grid's y)
    if (mb == 1) return launch_wide_mb<QT, AT, 1, F32, ROWS>(x, w, bias, y, M, N, K, s, st);
    if (mb == 2) return launch_wide_mb<QT, AT, 2, F32, ROWS>(x, w, bias, y, M, N, K, s, st);
    if constexpr (!F32) {
        if (mb == 3) return launch_wide_mb<QT, AT, 3, F32, ROWS>(x, w, bias, y, M, N, K, s, st);
        if (mb == 4) return launch_wide_mb<QT, AT, 4, F32, ROWS>(x, w, bias, y, M, N, K, s, st);
    }
    return -7;
}

template <int QT>
int launch_wide_q(const void *x, const void *w, const void *bias, void *y, int layout, int dt, int M, int N, int K, const WideShape &s,
                  hipStream_t st) {
    const bool rows = layout == LAYOUT_GGML;
    if (dt == DT_F16) return rows ? launch_wide_t<QT, _Float16, false, true>(x, w, bias, y, M, N, K, s, st)
                                  : launch_wide_t<QT, _Float16, false, false>(x, w, bias, y, M, N, K, s, st);
    if (dt == DT_BF16) return rows ? launch_wide_t<QT, __bf16, false, true>(x, w, bias, y, M, N, K, s, st)
                                   : launch_wide_t<QT, __bf16, false, false>(x, w, bias, y, M, N, K, s, st);
    if (dt == DT_F32) return rows ? launch_wide_t<QT, __bf16, true, true>(x, w, bias, y, M, N, K, s, st)
                                  : launch_wide_t<QT, __bf16, true, false>(x, w, bias, y, M, N, K, s, st);
    return -4;
}

template <int QT, typename AT, int MB>
static int launch_wide_mlp_mb(const void *x, const void *wg, const void *wu, void *y, int M, int N, int K, int act, const WideShape &s,
                              hipStream_t st) {
    if (s.r == 1) return launch_wide_r<QT, AT, MB, 1, false, false, true>(x, wg, wu, nullptr, y, M, N, K, act, s.waves, st);
    if constexpr (wide_mlp_two_rows(QT, __is_same(AT, _Float16), MB))
        if (s.r == 2) return launch_wide_r<QT, AT, MB, 2, false, false, true>(x, wg, wu, nullptr, y, M, N, K, act, s.waves, st);
    return -7;
}

// y = act(x wg^T) * (x wu^T), s.mb 16-row blocks of x to a workgroup (0: all of up to 64 rows)
template <int QT, typename AT>
static int launch_wide_mlp_t(const void *x, const void *wg, const void *wu, void *y, int M, int N, int K, int act, const WideShape &s,
                             hipStream_t st) {
    const int mb = s.mb ? s.mb : (M + 15) / 16;
    if (M > 16 * mb * 65535) return -7;                      // (blocks of rows are counted in the grid's y)
    if (mb == 1) return launch_wide_mlp_mb<QT, AT, 1>(x, wg, wu, y, M, N, K, act, s, st);
    if (mb == 2) return launch_wide_mlp_mb<QT, AT, 2>(x, wg, wu, y, M, N, K, act, s, st);
    if (mb == 3) return launch_wide_mlp_mb<QT, AT, 3>(x, wg, wu, y, M, N, K, act, s, st);
    return mb == 4 ? launch_wide_mlp_mb<QT, AT, 4>(x, wg, wu, y, M, N, K, act, s, st) : -7;
}

template <int QT>
int launch_wide_mlp_q(const void *x, const void *wg, const void *wu, void *y, int dt, int M, int N, int K, int act, const WideShape &s,
                      hipStream_t st) {
    if (dt == DT_F16) return launch_wide_mlp_t<QT, _Float16>(x, wg, wu, y, M, N, K, act, s, st);
    if (dt == DT_BF16) return launch_wide_mlp_t<QT, __bf16>(x, wg, wu, y, M, N, K, act, s, st);
    return -4;
}

}  // namespace lowbit
