// The gradient that flows on below a low-bit linear: gx[M,K] = g[M,N] * dequant(W)[N,K], from the packed tiled weight.
//
// Takes the place of dequantizing all of W to 16 bits and a dense product (low_bit_linear.py:519-541): same weights - one
// rounding of the fp32 value to the activation type - same 16-bit operands, fp32 sums, one rounding of the result.
//
// The sum runs along N, across the rows of the tiles, while a lane's 16 bytes of a tile are eight columns of one row: the
// operand of v_mfma_f32_32x32x16 needs the transpose.  So each wave turns one 16 x 128 tile per 64-row step into scaled 16-bit
// weights, writes them to LDS row by row, and all waves read them back with ds_read_b64_tr_b16, which hands lane i of
// 16 lanes element i of four rows.  g lies in LDS as the forward GEMM's x does.
//
// A workgroup owns 64 * MBW rows of g by 128 columns of gx: two groups of four waves, the first on the first half of the
// steps, the second on the rest, each with its own LDS buffers (two of each operand); their sums meet in LDS at the end.
// Within a group a wave owns all the rows by 32 columns.  What a step needs is loaded three steps ahead, into three sets of
// registers, and goes to LDS during the step before it.  (g by LDS-DMA instead, which the compiler does not count among
// the loads in flight, made it wait for the youngest ones and an earlier version a seventh slower.)
//
// What bounds it, 128 rows on [4096 x 4096] in sym_int4 (unsplit 33.7 us in a kernel trace, 1.05 us a pair of steps; split 15.9
// and 4.0 for the sums): LDS is busy 54 % of the time, the MFMA pipes 38 %, the vector units 30 %; two waves per SIMD that meet
// at a barrier per step overlap them badly.
// Of an earlier version's 39 us the MFMAs were 2, the dequantization with its writes to LDS 12, g's way into LDS 10.  64 rows
// by 64 columns per wave, whose operands are a fifth less LDS traffic, and the writes ahead of the MFMAs are level with this.
// Few tiles leave CUs idle: then several workgroups share a tile's walk (back_plan).
#include "lowbit_gemm.h"
#include "lowbit_splits.h"

namespace lowbit {

typedef short s16x4 __attribute__((ext_vector_type(4)));

__device__ inline f32x16 mfma32(f16x8 a, f16x8 b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0); }
__device__ inline f32x16 mfma32(bf16x8 a, bf16x8 b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }

constexpr int BACK_N = 64;                                   // weight rows per step
constexpr int BACK_WBYTES = BACK_N * TILE_COLS * 2;          // of scaled weights in LDS per step

// ws != null: workgroup (tile, s) walks the steps s * split_steps .. of N only and leaves its fp32 sums there for
// back_reduce_kernel.
template <int QT, typename AT, int MBW>
__global__ __launch_bounds__(512, 2) void gemm_back_kernel(const AT *__restrict__ g, const uint8_t *__restrict__ w,
                                                           AT *__restrict__ gx, int M, int N, int K, f32x4 *__restrict__ ws,
                                                           int split_steps) {
    using F = Fmt<QT>;
    using V8 = typename Vec8<AT>::type;
    constexpr int BM = 64 * MBW, GBYTES = BM * BACK_N * 2, GROUP = 2 * (GBYTES + BACK_WBYTES);
    __shared__ __attribute__((aligned(16))) uint8_t lds[2 * GROUP];
    const int lane = threadIdx.x & 63;
    const int wave_wg = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), half = wave_wg >> 2, wave = wave_wg & 3;

    const uint32_t grid_x = gridDim.x, splits = gridDim.y;
    // (one wait for all arguments: left alone the compiler loads each where it is first used, a scalar load's time apiece)
    asm volatile("" :: "s"(g), "s"(w), "s"(M), "s"(N), "s"(K), "s"(ws), "s"(split_steps), "s"(grid_x), "s"(splits));

    // Workgroups go to the XCDs in turn (id % 8): each takes a run of the tiles, the row tiles of a column tile side by side,
    // so that its L2 serves a column's weights to all of them.
    const int tiles_m = (M + BM - 1) / BM, G = K / TILE_COLS;
    // (What is dealt is tiles times splits, a tile's side by side: with an eighth of the tiles in every split the XCDs differ by up to
    // as many workgroups as there are splits, and those above a workgroup per CU wait.  125 rows on [9104 x 6272] in sym_int8, a
    // training step with the forward's splits dealt likewise: 89 -> 65 us.)
    const uint32_t units = (uint32_t)(tiles_m * G * splits), xcd = blockIdx.x & 7;           // (2^28 at most, see launch_back_m)
    const uint32_t unit = (units * xcd >> 3) + (blockIdx.x >> 3) + blockIdx.y * (grid_x >> 3);
    if (unit >= units * (xcd + 1) >> 3) return;              // whole workgroup leaves
    int tile = (int)unit, split = 0;
    if (ws) {
        tile = (int)(unit / splits);
        split = (int)(unit - tile * splits);
    }
    const int m0 = tile % tiles_m * BM, kt = tile / tiles_m;

    const int all_steps = (N + BACK_N - 1) / BACK_N, split_s0 = ws ? split * split_steps : 0;
    const int steps = ws && split_steps < all_steps - split_s0 ? split_steps : all_steps - split_s0, steps_first = (steps + 1) / 2;
    const int s0 = split_s0 + (half ? steps_first : 0), S = half ? steps - steps_first : steps_first, last = S > 0 ? S - 1 : 0;
    const int row_tiles = N / TILE_ROWS;
    // which step of the whole walk; past this group's last one: a re-read that nobody uses (a group may have no step at all)
    auto step_at = [&](int s) __attribute__((always_inline)) {
        s = s0 + (s < last ? s : last);
        return s < split_s0 + steps ? s : split_s0 + steps - 1;
    };

    // ---- the weights: this wave's tile of a step
    const int r16 = lane & 15, c4 = lane >> 4;
    const DqCtx ctx = {nullptr, dq_magic<QT, AT>()};
    uint32_t k04, k0123;
    asm("v_mov_b32 %0, 0x04040404" : "=v"(k04));
    asm("v_mov_b32 %0, 0x03020100" : "=v"(k0123));
    Nf4Scaled<AT> nf4;
    // 64-byte unit u (a sub-block) of row n lies at unit u ^ n % 4, its 16-byte chunk c at c ^ n / 4 % 4: the sixteen rows that a
    // write stores and the four rows by 64 bytes that a transposing read takes then cover all banks
    uint8_t *const wpos = lds + (wave * 16 + r16) * 256 + ((c4 ^ (r16 >> 2)) * 16);
    // scaled weights of sub-block j of t into the buffer at byte `at` of lds
    auto put_w = [&](const TileRegs<QT> &t, int j, int at) __attribute__((always_inline)) {
        u32x4 v;
        if constexpr (QT == QT_NF4) {
            if ((j & 1) == 0) {
#pragma unroll
                for (int q = 0; q < 4; q++)
#pragma unroll
                    for (int part = 0; part < 3; part++) nf4.build(t.h[0], j >> 1, q, part);
                nf4.take_built();
            }
#pragma unroll
            for (int u = 0; u < 8; u++) nf4.unit(t.q0[j], u, v, k04, k0123);
        } else {
#pragma unroll
            for (int p = 0; p < 4; p++) v[p] = Dequant<QT, AT>::pair(t, j, p, ctx);
        }
        *(u32x4 *)(wpos + at + ((j ^ (r16 & 3)) * 64)) = v;
    };

    // ---- g: through registers into pieces of 8 rows x 128 bytes, as the forward GEMM lays out x (row r = s ^ t % 2 of piece t and chunk
    // c' ^ r for lane 8 s + c'); wave w fills the 2 * MBW pieces from 2 * MBW * w on.  Rows past M read its last one.
    constexpr int PW = 2 * MBW;
    uint32_t goff[PW];                                       // bytes from the tile's first row, without the chunk
    uint32_t gchunk[2];                                      // 16-byte chunk in even and odd pieces
#pragma unroll
    for (int p = 0; p < 2; p++) gchunk[p] = (uint32_t)((lane & 7) ^ ((lane >> 3) ^ p));
#pragma unroll
    for (int j = 0; j < PW; j++) {
        int row = 8 * (PW * wave + j) + ((lane >> 3) ^ (j & 1));
        row = m0 + row < M ? row : M - 1 - m0;
        goff[j] = (uint32_t)row * (uint32_t)N * 2u;
    }
    const gbytes gbase = (gbytes)(const uint8_t *)g + (int64_t)m0 * N * 2;
    uint8_t *const gpos = lds + wave * PW * 1024 + lane * 16;
    struct Loads {
        TileRegs<QT> w;
        u32x4 g[PW];
    };
    auto load = [&](int s, Loads &t) __attribute__((always_inline)) {
        s = step_at(s);
        const gbytes src = gbase + (int64_t)s * (BACK_N * 2);
        const uint32_t chunks = (uint32_t)(N - s * BACK_N < BACK_N ? N - s * BACK_N : BACK_N) / 8;   // (columns past N: the row's last ones)
#pragma unroll
        for (int j = 0; j < PW; j++) {
            const uint32_t c = gchunk[j & 1];
            t.g[j] = ld<u32x4>(src + (goff[j] + (c < chunks ? c : chunks - 1) * 16u));
        }
        s = s * 4 + wave;
        s = s < row_tiles ? s : row_tiles - 1;               // rows past N: never multiplied
        load_tile<QT>((gbytes)w + ((int64_t)s * G + kt) * F::TILE_BYTES, lane, r16, t.w);
    };
    auto put_g = [&](const Loads &t, int j, int at) __attribute__((always_inline)) { *(u32x4 *)(gpos + at + j * 1024) = t.g[j]; };

    // ---- operands
    const int kg = lane >> 5, i32 = lane & 31;
    constexpr int RB = 2 * MBW;                              // 32-row blocks of g
    const uint8_t *const gread = lds + (i32 >> 3) * 1024 + (((i32 & 7) ^ ((i32 >> 3) & 1)) * 8) * 16;
    auto read_g = [&](int at, int ks, int mb) __attribute__((always_inline)) {
        return *(const V8 *)(gread + at + mb * 4096 + ((2 * ks + kg) ^ (i32 & 7)) * 16);
    };
    const int l16 = lane & 15, row4 = l16 >> 2, ch = ((lane >> 4) & 1) * 2 + ((l16 & 3) >> 1);
    uint8_t *const wread = lds + (8 * kg + row4) * 256 + (l16 & 1) * 8;
    auto read_w = [&](int at, int ks) __attribute__((always_inline)) {
        const int unit = (wave ^ row4) * 64;                 // this wave's 32 columns
        typedef short s16x8 __attribute__((ext_vector_type(8)));
        s16x8 v;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            uint8_t *p = wread + at + (16 * ks + 4 * h) * 256 + unit + ((ch ^ ((2 * kg + h) & 3)) * 16);
            const s16x4 q = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)p);
#pragma unroll
            for (int e = 0; e < 4; e++) v[h * 4 + e] = q[e];
        }
        return __builtin_bit_cast(V8, v);
    };

    f32x16 acc[RB];
#pragma unroll
    for (int mb = 0; mb < RB; mb++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc[mb][i] = 0.0f;

    const int w0 = half * GROUP, w1 = w0 + BACK_WBYTES, g0 = w1 + BACK_WBYTES, g1 = g0 + GBYTES;
    Loads ta, tb, tc;
    load(0, ta);
    load(1, tb);
    load(2, tc);
#pragma unroll
    for (int j = 0; j < PW; j++) put_g(ta, j, g0);
#pragma unroll
    for (int j = 0; j < 4; j++) put_w(ta.w, j, w0);
    __syncthreads();
    // Step s: what `ready` holds of step s + 1 goes to the other buffers, step s + 3 is loaded into the registers that step
    // s - 1 has freed.
    auto step = [&](int s, int wcur, int wnxt, int gcur, int gnxt, const Loads &ready, Loads &next, auto whole) __attribute__((always_inline)) {
        const int rest = N - (s0 + s) * BACK_N;              // a last step of 16, 32 or 48 rows
        V8 a[2], b[2][RB];
        auto read = [&](int ks) __attribute__((always_inline)) {
            a[ks & 1] = read_w(wcur, ks);
#pragma unroll
            for (int mb = 0; mb < RB; mb++) b[ks & 1][mb] = read_g(gcur, ks, mb);
        };
        read(0);
        __builtin_amdgcn_sched_barrier(0);
        load(s + 3, next);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int ks = 0; ks < 4; ks++) {
            if (ks < 3) read(ks + 1);                        // (rows past N: what is there, never multiplied)
            __builtin_amdgcn_sched_barrier(0);
            if (decltype(whole)::value || ks == 0 || ks * 16 < rest) {
#pragma unroll
                for (int mb = 0; mb < RB; mb++) acc[mb] = mfma32(a[ks & 1], b[ks & 1][mb], acc[mb]);
            }
            put_w(ready.w, ks, wnxt);
            if (ks < PW) put_g(ready, ks, gnxt);
            __builtin_amdgcn_sched_barrier(0);
        }
        __syncthreads();
    };
    // Two buffers, three sets of registers: a period of six.  The last one to six steps stand apart: one of them may hold fewer
    // rows, and a way out in the middle of the loop would make the compiler wait for loads at its head.
    typedef std::true_type whole_t;
    typedef std::false_type any_t;
    int s = 0;
    for (; s + 6 < S; s += 6) {
        step(s, w0, w1, g0, g1, tb, ta, whole_t());
        step(s + 1, w1, w0, g1, g0, tc, tb, whole_t());
        step(s + 2, w0, w1, g0, g1, ta, tc, whole_t());
        step(s + 3, w1, w0, g1, g0, tb, ta, whole_t());
        step(s + 4, w0, w1, g0, g1, tc, tb, whole_t());
        step(s + 5, w1, w0, g1, g0, ta, tc, whole_t());
    }
    if (s < S) {
        step(s, w0, w1, g0, g1, tb, ta, any_t());
        if (s + 1 < S) {
            step(s + 1, w1, w0, g1, g0, tc, tb, any_t());
            if (s + 2 < S) {
                step(s + 2, w0, w1, g0, g1, ta, tc, any_t());
                if (s + 3 < S) {
                    step(s + 3, w1, w0, g1, g0, tb, ta, any_t());
                    if (s + 4 < S) {
                        step(s + 4, w0, w1, g0, g1, tc, tb, any_t());
                        if (s + 5 < S) step(s + 5, w1, w0, g1, g0, ta, tc, any_t());
                    }
                }
            }
        }
    }
    for (int i = S; i < steps_first; i++) __syncthreads();   // the barrier of a step that the second group has not
    __syncthreads();

    // The groups' sums meet: the first keeps the first half of the row blocks, the second the others; each hands over what it
    // does not keep and stores the rest.
    f32x4 *const part = (f32x4 *)lds + wave * (RB * 256) + lane;
    auto give = [&](int from) __attribute__((always_inline)) {
#pragma unroll
        for (int mb = from; mb < from + MBW; mb++)
#pragma unroll
            for (int q = 0; q < 4; q++)
                part[(mb * 4 + q) * 64] = f32x4{acc[mb][q * 4], acc[mb][q * 4 + 1], acc[mb][q * 4 + 2], acc[mb][q * 4 + 3]};
    };
    // C layout: lane = 32 * kg + row of g, register i = column 8 * (i / 4) + 4 * kg + i % 4
    auto finish = [&](int from) __attribute__((always_inline)) {
        if (ws) {
            f32x4 *const to = ws + (((int64_t)split * (tiles_m * G) + tile) * 8 + wave_wg) * (MBW * 256) + lane;
#pragma unroll
            for (int mb = from; mb < from + MBW; mb++)
#pragma unroll
                for (int q = 0; q < 4; q++)
                    to[((mb - from) * 4 + q) * 64] = part[(mb * 4 + q) * 64] +
                        f32x4{acc[mb][q * 4], acc[mb][q * 4 + 1], acc[mb][q * 4 + 2], acc[mb][q * 4 + 3]};
            return;
        }
#pragma unroll
        for (int mb = from; mb < from + MBW; mb++) {
            const int m = m0 + mb * 32 + i32;
            AT *const row = gx + (int64_t)(m < M ? m : 0) * K + kt * TILE_COLS + wave * 32 + 4 * kg;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const f32x4 v = part[(mb * 4 + q) * 64];
                typedef AT at4 __attribute__((ext_vector_type(4)));
                at4 o;
#pragma unroll
                for (int t = 0; t < 4; t++) o[t] = to_at<AT>(acc[mb][q * 4 + t] + v[t]);
                if (m < M) *(at4 *)(row + 8 * q) = o;
            }
        }
    };
    if (half) give(0);
    else give(MBW);
    __syncthreads();
    if (half) finish(MBW);
    else finish(0);
}

// Adds the partial sums of the splits (as gemm_back_kernel leaves them: split, tile, wave, row block, register group, lane) in
// order and rounds once.  One thread per group of four columns.
template <typename AT, int MBW>
__global__ __launch_bounds__(256) void back_reduce_kernel(const f32x4 *__restrict__ ws, AT *__restrict__ gx, int M, int K, int64_t per_split,
                                                          int splits) {
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;           // (a split's sums are whole blocks of threads)
    const int lane = threadIdx.x & 63, q = threadIdx.x >> 6, mb = (int)(blockIdx.x % MBW), tw = (int)(blockIdx.x / MBW);
    const int wave_wg = tw & 7, tiles_m = (M + 64 * MBW - 1) / (64 * MBW);
    const int m = (tw >> 3) % tiles_m * (64 * MBW) + ((wave_wg >> 2) * MBW + mb) * 32 + (lane & 31);
    const int k = (tw >> 3) / tiles_m * TILE_COLS + (wave_wg & 3) * 32 + 8 * q + 4 * (lane >> 5);
    const f32x4 a = sum_splits(ws + t, per_split, splits);
    typedef AT at4 __attribute__((ext_vector_type(4)));
    at4 o;
#pragma unroll
    for (int i = 0; i < 4; i++) o[i] = to_at<AT>(a[i]);
    if (m < M) *(at4 *)(gx + (int64_t)m * K + k) = o;
}

// Tiles of gx with 64 or 128 rows each.
static int64_t back_tiles(int M, int K, int rows) { return (int64_t)((M + rows - 1) / rows) * (K / TILE_COLS); }

// How the tiles are cut: what takes the shortest by the estimate below, while the workgroups are one per CU at most (a workgroup's
// LDS fills a CU).  Where the result has fewer tiles than the GPU CUs, several workgroups share a tile's walk along N.
// Estimated microseconds, fitted to 258 random sizes (M = 24 .. 2048, N = 1024 .. 14336, K = 1024 .. 8192, five formats, both
// types) with up to 16 splits each: 6 % rms, the plan it picks within 2 % of the best on average.  A pair of steps takes 0.78
// (64 rows) or 1.03 (128), a launch 4.7 or 6.2, a second one that adds the splits 1.0 and 0.021 per 64 rows by 128 columns of fp32
// sums.  Splits are charged 12 instead of that 1.0: their workspace and launch cost the host 6, and where the GPU waits for the host
// anyway a step with them is the longer one (498 rows on [2000 x 1280] 42 -> 49, its kernel 18 -> 13).  Whole training steps against the choice without
// splits, us: 307 rows on [3360 x 1408] in nf4 65 -> 51, 234 on [7616 x 2432] 77 -> 50, 329 on [11456 x 4224] 168 -> 128, 125 on
// [9104 x 6272] in sym_int8 104 -> 89 (65 with this kernel's and the forward's splits dealt evenly to the XCDs); the kernels alone
// 1.34 times as fast over those 258 sizes, 0.90 at worst.
struct BackPlan {
    int rows, splits;             // rows of g per tile; workgroups that share a tile's walk along N
};
static double back_time_us(int qtype, int64_t tiles, int rows, int N, int splits) {
    const int steps = (N + BACK_N - 1) / BACK_N, per = (steps + splits - 1) / splits;
    const double format = qtype == QT_NF4 ? 1.2 : qtype == QT_SYM_INT4 || qtype == QT_ASYM_INT4 ? 1.06 : 0.99;
    const double t = (rows == 64 ? 4.7 : 6.2) + (rows == 64 ? 0.78 : 1.03) * format * ((per + 1) / 2);
    return splits > 1 ? t + 12.0 + 0.021 * (double)splits * (double)tiles * rows / 64 : t;
}
static size_t back_split_bytes(int M, int K, int rows) { return (size_t)back_tiles(M, K, rows) * rows * TILE_COLS * sizeof(float); }

static BackPlan back_plan(int qtype, int M, int N, int K, size_t ws_bytes) {
    const int steps = (N + BACK_N - 1) / BACK_N;
    BackPlan best = {128, 1};
    double best_us = 1e30;
    auto consider = [&](int rows, int s) {
        const double us = back_time_us(qtype, back_tiles(M, K, rows), rows, N, s);
        if (us < best_us) {
            best = {rows, s};
            best_us = us;
        }
    };
    for (int rows = 64; rows <= 128; rows += 64)
        if (back_tiles(M, K, rows) <= 256) consider(rows, 1);
    if (best_us < 18.0) return best;                         // (no split is estimated shorter)
    for (int rows = 64; rows <= 128; rows += 64)
        for (int s = 2; s <= 16 && back_tiles(M, K, rows) * s <= 256 && 2 * s <= steps && s * back_split_bytes(M, K, rows) <= ws_bytes; s++)
            if ((steps + s - 1) / s < (steps + s - 2) / (s - 1)) consider(rows, s);        // (fewer steps than with one split less)
    return best;
}

size_t back_workspace_bytes(int qtype, int M, int N, int K) {
    const BackPlan p = back_plan(qtype, M, N, K, (size_t)-1);
    return p.splits > 1 ? (size_t)p.splits * back_split_bytes(M, K, p.rows) : 0;
}

template <int QT, typename AT, int MBW>
static int launch_back_m(const void *g, const void *w, void *gx, int M, int N, int K, int splits, void *ws, hipStream_t st) {
    const int64_t tiles = back_tiles(M, K, 64 * MBW);
    if (tiles > (1 << 28)) return -3;
    const int steps = (N + BACK_N - 1) / BACK_N, per = (steps + splits - 1) / splits, ny = (steps + per - 1) / per;
    if (ny == 1) ws = nullptr;
    hipLaunchKernelGGL((gemm_back_kernel<QT, AT, MBW>), dim3(8 * (unsigned)((tiles + 7) / 8), ny), dim3(512), 0, st, (const AT *)g,
                       (const uint8_t *)w, (AT *)gx, M, N, K, (f32x4 *)ws, per);
    if (ws) {
        const int64_t per_split = tiles * 8 * MBW * 256;                 // groups of four sums
        hipLaunchKernelGGL((back_reduce_kernel<AT, MBW>), dim3((unsigned)(per_split / 256)), dim3(256), 0, st, (const f32x4 *)ws, (AT *)gx,
                           M, K, per_split, ny);
    }
    return 0;
}

template <int QT, typename AT>
static int launch_back_t(const void *g, const void *w, void *gx, int M, int N, int K, void *ws, size_t ws_bytes, hipStream_t st) {
    const BackPlan p = back_plan(QT, M, N, K, ws ? ws_bytes : 0);
    if (p.rows == 128) return launch_back_m<QT, AT, 2>(g, w, gx, M, N, K, p.splits, ws, st);
    return launch_back_m<QT, AT, 1>(g, w, gx, M, N, K, p.splits, ws, st);
}

template <int QT>
static int launch_back_q(const void *g, const void *w, void *gx, int dt, int M, int N, int K, void *ws, size_t ws_bytes, hipStream_t st) {
    if (dt == DT_F16) return launch_back_t<QT, _Float16>(g, w, gx, M, N, K, ws, ws_bytes, st);
    if (dt == DT_BF16) return launch_back_t<QT, __bf16>(g, w, gx, M, N, K, ws, ws_bytes, st);
    return -4;
}

// Whether this kernel is the faster way, against dequantizing W and torch's dense product: while its tiles of 128 rows are one per
// CU at most (with a second round it is 0.6 - 1.3 times as fast), and there are 20 workgroups or more.  A K below 1024 leaves few
// column tiles, and there the walk along N is to be no longer than four times K over 20 tiles at least.  Over 1150 random sizes, M =
// 200 .. 2048, N = 4096 .. 152000, K = 1024 .. 8192: shared walks 1.8 times as fast and never slower, tiles of 64 rows 1.17 (11 of
// 180 slower by more than 3 %), unshared tiles of 128 rows
//   - 1.2 in fp8_e4m3, never slower, and 1.07 in the integers where N is more than four times K (1.2 below): 28 of 111 are slower by
//     more than 3 %, 0.78 at worst, because the dense product's rate varies from 320 to 830 TFLOP/s between neighbouring sizes;
//   - in nf4, which takes 1.2 of the others' time, 1.06 up to N = 2.5 K and 0.98 beyond (187 of 336 slower by more than 3 %, 0.69 at
//     worst; 1064 rows on [13984 x 2816] 153 us against 137): not taken there.
// With less workspace than the plan asks for the walks are longer: then it is the faster way from 20 tiles on while N is no longer than
// twice K, and from 80 on up to four times (4900 random sizes, 1.64 times as fast on average, 31 more than 5 % slower, 0.79 at worst).
bool gemm_back_applies(int qtype, int M, int N, int K, size_t ws_bytes) {
    BackPlan p = back_plan(qtype, M, N, K, (size_t)-1);
    const bool shared = p.splits == 1 || (size_t)p.splits * back_split_bytes(M, K, p.rows) <= ws_bytes;
    if (!shared) p = back_plan(qtype, M, N, K, 0);
    const int64_t tiles = back_tiles(M, K, p.rows);
    if (tiles > 256 || N >= (1 << 23)) return false;
    if (!shared) return N <= 2 * (int64_t)K ? tiles >= 20 : qtype != QT_NF4 && tiles >= 80 && N <= 4 * (int64_t)K;
    if (K < 1024) return tiles >= 20 && N <= (qtype == QT_NF4 ? 2 : 4) * (int64_t)K;
    if (qtype == QT_NF4 && p.rows == 128 && p.splits == 1 && 2 * (int64_t)N > 5 * (int64_t)K) return false;
    return tiles * p.splits >= 20;
}

// gx[M, K] = g[M, N] * dequant(w)[N, K]; w tiled, g and gx 16-byte aligned, N below 2^23 (32-bit offsets within a row tile)
int launch_gemm_back(const void *g, const void *w, void *gx, int qtype, int act_dtype, int M, int N, int K, void *ws, size_t ws_bytes,
                     hipStream_t st) {
    if (M == 0 || K == 0) return 0;
    if (N >= (1 << 23)) return -3;
    switch (qtype) {
    case QT_SYM_INT4: return launch_back_q<QT_SYM_INT4>(g, w, gx, act_dtype, M, N, K, ws, ws_bytes, st);
    case QT_ASYM_INT4: return launch_back_q<QT_ASYM_INT4>(g, w, gx, act_dtype, M, N, K, ws, ws_bytes, st);
    case QT_SYM_INT8: return launch_back_q<QT_SYM_INT8>(g, w, gx, act_dtype, M, N, K, ws, ws_bytes, st);
    case QT_NF4: return launch_back_q<QT_NF4>(g, w, gx, act_dtype, M, N, K, ws, ws_bytes, st);
    case QT_FP8_E4M3: return launch_back_q<QT_FP8_E4M3>(g, w, gx, act_dtype, M, N, K, ws, ws_bytes, st);
    default: return -2;
    }
}

}  // namespace lowbit
