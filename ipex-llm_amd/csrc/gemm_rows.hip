// Batches of more than 16 rows against weights in the row-major (ggml) layout, any shape: y[M,N] = x[M,K] dequant(W)[N,K]^T.
//
// Untileable weights (out_features no multiple of 16 or in_features no multiple of 128) had the streaming kernel only: a
// pass over the weights per 16 rows of x.  Here a workgroup of four waves owns 16 * MB rows of x by 128 weight
// rows; its waves split the weight rows, share the block of x in LDS (two buffers, one 128-column step of prefetch
// through registers) and use every unpacked weight for all rows.
//
// The operands are those of lowbit_rows.h: exact codes, and the block scale applied to the fp32 result of each
// v_mfma_f32_16x16x32, so nothing of a weight is rounded to 16 bits.  That scale is what bounds it: one FMA per result
// and 32 columns (asym_int4: three operations) is as much vector time as the MFMA takes matrix time, and unpacking adds to
// it - the reason for many rows of x per unpacked weight (MB = 8) where M allows.  333 rows on [3200 x 8640], 272 us as 21
// streaming passes in sym_int4: 51.6 us with the reduction (357 TFLOP/s) in sym_int4, 67 in asym_int4, 70 (fp16) and 85
// (bf16, three MFMAs per step) in nf4, 55 in sym_int8, 49 in fp8_e4m3 ([3201 x 8704]).
#include "lowbit_mfma.h"
#include "lowbit_rows.h"
#include "lowbit_unpack.h"

namespace lowbit {

int launch_gemv(const void *x, const void *w, const void *bias, void *y, int qtype, int layout, int act_dtype, int M, int N, int K,
                int waves, hipStream_t st);

constexpr int RG_WAVES = 4, RG_NB = 2, RG_N = RG_WAVES * RG_NB * TILE_ROWS;      // 128 weight rows per workgroup

// MB: 16-row blocks of x per workgroup.  blockIdx.y: the K split, whose partial sums go to ws in register order.
template <int QT, typename AT, int MB>
__global__ __launch_bounds__(256, 2) void gemm_rows_kernel(const AT *__restrict__ x, const uint8_t *__restrict__ w,
                                                           const AT *__restrict__ bias, AT *__restrict__ y, int M, int N, int K,
                                                           int steps, float *__restrict__ ws) {
    using F = Fmt<QT>;
    using V8 = typename Vec8<AT>::type;
    using Op = Operand<QT, AT, false, true>;
    constexpr float OFFSET = Op::OFFSET;
    constexpr bool NEED_S = Op::NEED_S;
    constexpr int PARTS = Op::PARTS;
    constexpr int BM = 16 * MB, NB = RG_NB;
    __shared__ __attribute__((aligned(16))) uint8_t xs[2][BM * 256];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, c = lane >> 4;

    // Workgroups go to the XCDs in turn (id % 8): each XCD takes a run of the tiles, row tile by row tile within a column
    // tile, so that its L2 serves a column's weights to all their row tiles.
    const int tiles_m = (M + BM - 1) / BM, tiles = tiles_m * ((N + RG_N - 1) / RG_N), per_xcd = (tiles + 7) / 8;
    const int tile = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if (tile >= tiles) return;                               // whole workgroup leaves
    const int m0 = tile % tiles_m * BM, n0 = tile / tiles_m * RG_N + wave * (NB * TILE_ROWS);

    const int blocks = K / F::QK, G = (K + TILE_COLS - 1) / TILE_COLS;
    const int g0 = blockIdx.y * steps, g1 = g0 + steps < G ? g0 + steps : G;
    gbytes wr[NB];
#pragma unroll
    for (int nb = 0; nb < NB; nb++) {
        const int n = n0 + nb * TILE_ROWS + r;
        wr[nb] = (gbytes)w + (int64_t)(n < N ? n : N - 1) * blocks * F::TS;
    }
    // this thread's chunks of the x block: 16 lanes per row
    const int u = threadIdx.x & 15, xrow = threadIdx.x >> 4;
    const uint8_t *const xtile = (const uint8_t *)(x + (int64_t)m0 * K);
    uint32_t xoff[MB];                                       // bytes from the tile's first row (K < 2^23)
#pragma unroll
    for (int i = 0; i < MB; i++) {
        const int m = i * 16 + xrow;
        xoff[i] = (uint32_t)(m0 + m < M ? m : M - 1 - m0) * (uint32_t)K * 2u;
    }
    auto load_x = [&](int g, u32x4 (&v)[MB]) __attribute__((always_inline)) {
        const int col = g * TILE_COLS + u * 8;
        const bool past = col >= K;                          // columns past K read as zero (from the row's first ones)
        const uint32_t at = past ? 0 : (uint32_t)col * 2u;
#pragma unroll
        for (int i = 0; i < MB; i++) {
            v[i] = *(const u32x4 *)(xtile + (xoff[i] + at));
            v[i] = past ? u32x4{0u, 0u, 0u, 0u} : v[i];
        }
    };
    auto load_w = [&](int g, RowRegs<QT> (&t)[NB]) __attribute__((always_inline)) {
#pragma unroll
        for (int nb = 0; nb < NB; nb++) load_rows<QT>(wr[nb], g, c, blocks, t[nb]);
    };
    auto put_x = [&](uint8_t *buf, const u32x4 (&v)[MB]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < MB; i++) store_x_rows<QT>(buf + (i * 16 + xrow) * 256, u, v[i], xrow);
    };

    f32x4 acc[MB][NB];
#pragma unroll
    for (int mb = 0; mb < MB; mb++)
#pragma unroll
        for (int nb = 0; nb < NB; nb++) acc[mb][nb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    const f32x4 zero4 = {0.0f, 0.0f, 0.0f, 0.0f};
    const V8 ones = ones8<AT>();
    const Op op;

    u32x4 xr[MB];
    RowRegs<QT> wc[NB], wn[NB];
    load_x(g0, xr);
    load_w(g0, wc);
    put_x(xs[0], xr);
    __syncthreads();
    for (int g = g0; g < g1; g++) {
        const uint8_t *cur = xs[(g - g0) & 1];
        const bool more = g + 1 < g1;
        if (more) {
            load_x(g + 1, xr);
            load_w(g + 1, wn);
        }
        uint32_t hb[NB][4];
#pragma unroll
        for (int nb = 0; nb < NB; nb++) arrange_rows<QT>(wc[nb], hb[nb]);
        // Unit q = (step j, 16-row block mb), in the order the hardware should issue them: the MFMAs of a unit, the LDS
        // read of the next one's x, then the scaling of the unit before, whose results have landed meanwhile.  Left
        // alone the scheduler issues the step's reads and MFMAs together and runs out of registers.
        auto read_x = [&](int q) __attribute__((always_inline)) {
            const int j = q / MB, mb = q % MB;
            return *(const V8 *)(cur + (mb * 16 + r) * 256 + (((j * 4 + c) ^ r) * 16));
        };
        V8 a = read_x(0), b[NB][PARTS];
        float d[2][NB], e[2][NB];                            // of this step and the one before
        f32x4 p[2][NB], sum[2];
#pragma unroll
        for (int q = 0; q <= 4 * MB; q++) {
            if (q < 4 * MB) {
                const int j = q / MB;
                if (q % MB == 0) {
#pragma unroll
                    for (int nb = 0; nb < NB; nb++) {
#pragma unroll
                        for (int part = 0; part < PARTS; part++) b[nb][part] = op.get(wc[nb], j, part);
                        float mn;
                        hdr_to_scale<QT>(hb[nb][j], d[j & 1][nb], mn);
                        e[j & 1][nb] = mn - OFFSET * d[j & 1][nb];
                        d[j & 1][nb] = Op::scale(d[j & 1][nb]);
                    }
                }
                if constexpr (NEED_S) sum[q & 1] = mfma16(a, ones, zero4);
#pragma unroll
                for (int nb = 0; nb < NB; nb++) p[q & 1][nb] = Op::product(a, a, b[nb]);
                if (q + 1 < 4 * MB) a = read_x(q + 1);
            }
            if (q > 0) {
                const int o = (q - 1) & 1, mb = (q - 1) % MB, j = (q - 1) / MB;
#pragma unroll
                for (int nb = 0; nb < NB; nb++)
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        acc[mb][nb][i] = Op::add(acc[mb][nb][i], d[j & 1][nb], p[o][nb][i], e[j & 1][nb], sum[o][i]);
#pragma unroll
                for (int nb = 0; nb < NB; nb++) asm volatile("" : "+v"(acc[mb][nb]));
            }
        }
        if (more) {
            put_x(xs[(g + 1 - g0) & 1], xr);
#pragma unroll
            for (int nb = 0; nb < NB; nb++) wc[nb] = wn[nb];
        }
        __syncthreads();
    }

    // C layout: lane = 16*grp + column (weight row), register i = row 4*grp + i of x
    if (ws) {
        f32x4 *part = (f32x4 *)ws + (((int64_t)blockIdx.y * tiles + tile) * RG_WAVES + wave) * (MB * NB * 64) + lane;
#pragma unroll
        for (int mb = 0; mb < MB; mb++)
#pragma unroll
            for (int nb = 0; nb < NB; nb++) part[(mb * NB + nb) * 64] = acc[mb][nb];
        return;
    }
#pragma unroll
    for (int nb = 0; nb < NB; nb++) {
        const int n = n0 + nb * TILE_ROWS + r;
        if (n >= N) continue;
        const float bv = bias ? (float)bias[n] : 0.0f;
        uint32_t again = 0;                                   // results that are not finite, see dot_fp32
#pragma unroll
        for (int mb = 0; mb < MB; mb++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int m = m0 + mb * 16 + c * 4 + i;
                if (m < M) {
                    y[(int64_t)m * N + n] = to_at<AT>(acc[mb][nb][i] + bv);
                    again |= __builtin_isfinite(acc[mb][nb][i]) ? 0u : 1u << (mb * 4 + i);
                }
            }
        for (; again; again &= again - 1) {
            const int bit = __builtin_ctz(again), m = m0 + bit / 4 * 16 + c * 4 + bit % 4;
            y[(int64_t)m * N + n] = to_at<AT>(dot_fp32<QT, true>(x + (int64_t)m * K, w, n, K) + bv);
        }
    }
}

// Sums the splits and writes y, rounded once: one thread per four rows of one column.
template <int QT, typename AT, int MB>
__global__ __launch_bounds__(256) void gemm_rows_reduce_kernel(const f32x4 *__restrict__ ws, const AT *__restrict__ x,
                                                               const uint8_t *__restrict__ w, const AT *__restrict__ bias,
                                                               AT *__restrict__ y, int M, int N, int K, int tiles, int splits) {
    constexpr int PER_TILE = RG_WAVES * MB * RG_NB * 64;     // a multiple of 256
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int tiles_m = (M + 16 * MB - 1) / (16 * MB);
    const int tile = (int)(t / PER_TILE), in = (int)(t % PER_TILE);
    const int lane = in & 63, nb = (in >> 6) % RG_NB, mb = (in >> 6) / RG_NB % MB, wave = (in >> 6) / (RG_NB * MB);
    const int m = tile % tiles_m * 16 * MB + mb * 16 + (lane >> 4) * 4;
    const int n = tile / tiles_m * RG_N + (wave * RG_NB + nb) * TILE_ROWS + (lane & 15);
    if (m >= M || n >= N) return;
    f32x4 a = ws[t];
    for (int s = 1; s < splits; s++) a += ws[(int64_t)s * tiles * PER_TILE + t];
    const float bv = bias ? (float)bias[n] : 0.0f;
#pragma unroll
    for (int i = 0; i < 4; i++)
        if (m + i < M) y[(int64_t)(m + i) * N + n] = to_at<AT>(a[i] + bv);
    for (int i = 0; i < 4; i++) {                            // results that are not finite, see dot_fp32
        const float sum = i == 0 ? a[0] : i == 1 ? a[1] : i == 2 ? a[2] : a[3];
        if (m + i < M && !__builtin_isfinite(sum))
            y[(int64_t)(m + i) * N + n] = to_at<AT>(dot_fp32<QT, true>(x + (int64_t)(m + i) * K, w, n, K) + bv);
    }
}

struct RowsPlan {
    int mb, tiles, steps, splits;
    size_t ws_bytes;
};
// Rows of x per workgroup: 128 where that pads M by little more than 64 would, fewer for small batches.  K splits:
// until the workgroups are about two per CU (the kernel's occupancy), of at least four steps each.
static RowsPlan rows_plan(int M, int N, int K, size_t ws_bytes) {
    RowsPlan p;
    const int pad64 = (M + 63) / 64 * 64, pad128 = (M + 127) / 128 * 128;
    p.mb = M <= 32 ? 2 : M <= 64 || pad128 * 8 > pad64 * 9 ? 4 : 8;
    p.tiles = ((M + 16 * p.mb - 1) / (16 * p.mb)) * ((N + RG_N - 1) / RG_N);
    const int G = (K + TILE_COLS - 1) / TILE_COLS;
    const size_t per_split = (size_t)p.tiles * 16 * p.mb * RG_N * sizeof(float);
    int s = 512 / p.tiles;
    s = s > G / 4 ? G / 4 : s;
    s = s > 16 ? 16 : s;
    while (s > 1 && (size_t)s * per_split > ws_bytes) s--;
    if (s < 1) s = 1;
    p.steps = (G + s - 1) / s;
    p.splits = (G + p.steps - 1) / p.steps;
    p.ws_bytes = p.splits > 1 ? p.splits * per_split : 0;
    return p;
}

size_t gemm_rows_workspace_bytes(int M, int N, int K, size_t max_bytes) { return rows_plan(M, N, K, max_bytes).ws_bytes; }

template <int QT, typename AT, int MB>
static void launch_rows_m(const void *x, const void *w, const void *bias, void *y, int M, int N, int K, const RowsPlan &p, float *ws,
                          hipStream_t st) {
    if (p.splits == 1) ws = nullptr;
    hipLaunchKernelGGL((gemm_rows_kernel<QT, AT, MB>), dim3((p.tiles + 7) / 8 * 8, p.splits), dim3(256), 0, st, (const AT *)x,
                       (const uint8_t *)w, (const AT *)bias, (AT *)y, M, N, K, p.steps, ws);
    if (ws)
        hipLaunchKernelGGL((gemm_rows_reduce_kernel<QT, AT, MB>), dim3((unsigned)((int64_t)p.tiles * RG_WAVES * MB * RG_NB * 64 / 256)),
                           dim3(256), 0, st, (const f32x4 *)ws, (const AT *)x, (const uint8_t *)w, (const AT *)bias, (AT *)y, M, N, K,
                           p.tiles, p.splits);
}

template <int QT, typename AT>
static int launch_rows_t(const void *x, const void *w, const void *bias, void *y, int M, int N, int K, const RowsPlan &p, float *ws,
                         hipStream_t st) {
    if (p.mb == 2) launch_rows_m<QT, AT, 2>(x, w, bias, y, M, N, K, p, ws, st);
    else if (p.mb == 4) launch_rows_m<QT, AT, 4>(x, w, bias, y, M, N, K, p, ws, st);
    else launch_rows_m<QT, AT, 8>(x, w, bias, y, M, N, K, p, ws, st);
    return 0;
}

template <int QT>
static int launch_rows_q(const void *x, const void *w, const void *bias, void *y, int dt, int M, int N, int K, const RowsPlan &p,
                         float *ws, hipStream_t st) {
    if (dt == DT_F16) return launch_rows_t<QT, _Float16>(x, w, bias, y, M, N, K, p, ws, st);
    if (dt == DT_BF16) return launch_rows_t<QT, __bf16>(x, w, bias, y, M, N, K, p, ws, st);
    return -4;
}

int launch_gemm_rows(const void *x, const void *w, const void *bias, void *y, int qtype, int act_dtype, int M, int N, int K,
                     void *workspace, size_t workspace_bytes, hipStream_t st) {
    if (M == 0 || N == 0) return 0;
    const RowsPlan p = rows_plan(M, N, K, workspace ? workspace_bytes : 0);
    if (K >= (1 << 23))                                      // 32-bit offsets within a tile of x: the streaming kernel has 64
        return launch_gemv(x, w, bias, y, qtype, LAYOUT_GGML, act_dtype, M, N, K, 0, st);
    if ((int64_t)((M + 15) / 16) * ((N + RG_N - 1) / RG_N) > 0x7ffffff) return -3;
    float *ws = (float *)workspace;
    switch (qtype) {
    case QT_SYM_INT4: return launch_rows_q<QT_SYM_INT4>(x, w, bias, y, act_dtype, M, N, K, p, ws, st);
    case QT_ASYM_INT4: return launch_rows_q<QT_ASYM_INT4>(x, w, bias, y, act_dtype, M, N, K, p, ws, st);
    case QT_SYM_INT8: return launch_rows_q<QT_SYM_INT8>(x, w, bias, y, act_dtype, M, N, K, p, ws, st);
    case QT_NF4: return launch_rows_q<QT_NF4>(x, w, bias, y, act_dtype, M, N, K, p, ws, st);
    case QT_FP8_E4M3: return launch_rows_q<QT_FP8_E4M3>(x, w, bias, y, act_dtype, M, N, K, p, ws, st);
    default: return -2;
    }
}

}  // namespace lowbit
