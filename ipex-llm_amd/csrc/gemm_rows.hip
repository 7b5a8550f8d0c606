// Batches of more than 16 rows against weights in the row-major (ggml) layout, any shape: y[M,N] = x[M,K] dequant(W)[N,K]^T.
//
// Untileable weights (out_features no multiple of 16 or in_features no multiple of 128) had the streaming kernel only: a
// pass over the weights per 16 rows of x.  Here a workgroup of four waves owns 32 * MB rows of x by 128 weight
// rows; its waves split the weight rows, share the block of x in LDS (two buffers, one 128-column step of prefetch
// by LDS-DMA) and use every unpacked weight for all rows.
//
// The operands are exact codes, and the block scale is applied to the fp32 result of a block's MFMAs, so nothing of a weight
// is rounded to 16 bits.  That scale bounds the formats with blocks of 32: 16 FMAs (asym_int4: 48 operations) to two
// v_mfma_f32_32x32x16, and the two do not overlap fully - an MFMA takes the issue of about 2.5 FMAs from either wave of a
// SIMD.  Hence the 32 x 32 form (half the MFMAs of 16 x 16 x 32 for the same work: 21.0 against 24.7 ns per 32768 products
// and 8 FMAs), one scaling per block of nf4 and fp8_e4m3 in place of one per 32 columns, and x by LDS-DMA in its own order: the
// weights are unpacked so that a lane's eight codes are eight consecutive columns, where before x was permuted on its way
// through registers.  The loads are spread over the step: 8 KB of LDS-DMA per wave over its first half, half of the weights at
// its head and half in the middle (fp8_e4m3: all in the middle, 5 - 15 % faster than with some at the head).  Everything at
// the head waits for each other, 7 % of the time in sym_int4 and 13 % in fp8_e4m3; all weights in the middle, the others
// lose 2 % on average and up to 8 where the weights come from HBM (180 rows on [27966 x 9696] in asym_int4 325 / 313 us).
// Left: the memory system (without the loads of x a step is 15 % shorter), and without FMAs, x and weights still 60 % of it.
// Eight waves on 256 weight rows, which halve x's traffic, gain 5 - 9 % on [8008 x 8256] and lose as much elsewhere.
// 333 rows on [3200 x 8640] with the reduction, 16 x 16 x 32 and x through registers / now: sym_int4 52.0 / 42.5 us (433
// TFLOP/s), asym_int4 67.3 / 64.7, sym_int8 56.3 / 48.6, nf4 70.4 / 59.8 (fp16, two MFMAs per product) and 85.9 / 73.4 (bf16,
// three), fp8_e4m3 51.2 / 38.9 ([3201 x 8704]); 2000 rows on [4001 x 4160] 115.2 / 92.1 in sym_int4, 125.4 / 107.1 in
// sym_int8; 1.23 times as fast on average over 1000 points, 3 of them slower by 5 to 8 %.
#include "lowbit_mfma.h"
#include "lowbit_rows.h"
#include "lowbit_splits.h"
#include "lowbit_unpack.h"

#include <type_traits>

namespace lowbit {

int launch_gemv(const void *x, const void *w, const void *bias, void *y, int qtype, int layout, int act_dtype, int M, int N, int K,
                int waves, hipStream_t st);

constexpr int RG_WAVES = 4, RG_N = RG_WAVES * 32;        // 128 weight rows per workgroup, 32 per wave
constexpr int RG_CUS = 256;                              // what the order of the splits reckons with

typedef float f32x16 __attribute__((ext_vector_type(16)));
__device__ inline f32x16 mfma32(f16x8 a, f16x8 b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0); }
__device__ inline f32x16 mfma32(bf16x8 a, bf16x8 b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }

// Codes and headers of 32 weight rows by 128 columns, in 16-byte pieces:
//   sym_int4, sym_int8  lane l = 16 * b + r holds block b of rows r and 16 + r (sym_int8: two pieces each), as the streaming
//                       kernel's lanes do: the loads that touch a row's lines then follow each other.  With 32 rows to a load
//                       and a block's half to a lane the lines of a wave's 32 rows, with four waves as much as the L1 holds,
//                       were often gone before the last load of them (sym_int8: 30 rows on [17069 x 9600] 89.6 us, now 66.4)
//   asym_int4           lane 32 * c + r: blocks c and 2 + c of row r (its scale leaves the vector units no time for twice the
//                       lane swaps: in sets 1 % slower over 600 points)
//   nf4                 lane 32 * c + r: half c of either block's 32 bytes of row r
//   fp8_e4m3            lane 32 * c + r: bytes 16c .. 16c+15 of each 32 columns of row r
template <int QT> struct RowRegs32 {
    static constexpr bool SETS = QT == QT_SYM_INT4 || QT == QT_SYM_INT8;       // pieces in two sets of 16 rows
    static constexpr int NQ = Fmt<QT>::BITS == 8 ? 4 : 2, NH = QT == QT_FP8_E4M3 ? 1 : 2;
    u32x4 q[NQ];
    uint32_t h[NH];
};
// row: the lane's weight row, SETS: those of either set.  Blocks past the end of the row are read from its last one (their
// scale is made zero).
template <int QT> __device__ inline void load_rows32(const gbytes (&row)[2], int g, int lane, int blocks, RowRegs32<QT> &t, int from = 0, int to = RowRegs32<QT>::NQ) {
    using F = Fmt<QT>;
    using R = RowRegs32<QT>;
    constexpr int PER = TILE_COLS / F::QK;                   // blocks per group of columns
    const int c = lane >> 5;
    auto block = [&](gbytes row, int i) __attribute__((always_inline)) {
        const int b = g * PER + i;
        return row + (int64_t)(b < blocks ? b : blocks - 1) * F::TS;
    };
    auto header = [&](gbytes p) __attribute__((always_inline)) -> uint32_t {
        if constexpr (F::HDR == 2) return *(const __attribute__((address_space(1))) uint16_t *)p;
        else return *(const __attribute__((address_space(1))) u32_a2 *)p;
    };
#pragma unroll
    for (int i = from; i < to; i++) {
        constexpr int EACH = R::NQ / 2;                      // SETS: pieces per set
        const gbytes p = R::SETS ? block(row[i / EACH], lane >> 4) + i % EACH * 16 : QT == QT_NF4 ? block(row[0], i) + 16 * c
                       : QT == QT_FP8_E4M3 ? block(row[0], 0) + 32 * i + 16 * c : block(row[0], 2 * i + c);
        if (R::SETS && i % EACH == 0) t.h[i / EACH] = header(p);
        t.q[i] = *(const __attribute__((address_space(1))) u32x4_a2 *)(p + F::HDR);
    }
    if constexpr (!R::SETS) {
        if (from > 0) return;                                // (the headers come with the first piece)
#pragma unroll
        for (int i = 0; i < R::NH; i++) t.h[i] = header(block(row[0], QT == QT_ASYM_INT4 ? 2 * i + c : i));
    }
}
// After this lane 32 * c + r has half c of sub-step j (32 columns) of row r in q[j / 2][2 * (j & 1)] and the next dword (4 bits) or
// in q[j] (8 bits), and its block's header in hb[j].
template <int QT> __device__ inline void arrange_rows32(RowRegs32<QT> &t, uint32_t (&hb)[4]) {
    if constexpr (QT == QT_FP8_E4M3) {
        hb[0] = hb[1] = hb[2] = hb[3] = t.h[0];
    } else if constexpr (QT == QT_NF4) {
        hb[0] = hb[1] = t.h[0];
        hb[2] = hb[3] = t.h[1];
    } else if constexpr (QT == QT_ASYM_INT4) {
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const auto h = __builtin_amdgcn_permlane32_swap(t.h[i], t.h[i], false, false);
            const auto a = __builtin_amdgcn_permlane32_swap(t.q[i][0], t.q[i][2], false, false);
            const auto b = __builtin_amdgcn_permlane32_swap(t.q[i][1], t.q[i][3], false, false);
            hb[2 * i] = h[0];
            hb[2 * i + 1] = h[1];
            t.q[i] = u32x4{a[0], b[0], a[1], b[1]};
        }
    } else {
        // the set changes places with bit 0 of the block, then the half (4 bits: dwords 0, 1 and 2, 3) with bit 1
        constexpr bool WIDE = Fmt<QT>::BITS == 8;
        const RowRegs32<QT> in = t;
#pragma unroll
        for (int d = 0; d < (WIDE ? 4 : 2); d++) {
            uint32_t m[2][2];                                // [block % 2][half]
#pragma unroll
            for (int half = 0; half < 2; half++) {
                const auto v = WIDE ? __builtin_amdgcn_permlane16_swap(in.q[half][d], in.q[WIDE ? 2 + half : 0][d], false, false)
                                    : __builtin_amdgcn_permlane16_swap(in.q[0][(2 * half + d) % 4], in.q[1][(2 * half + d) % 4], false, false);
                m[0][half] = v[0];
                m[1][half] = v[1];
            }
#pragma unroll
            for (int odd = 0; odd < 2; odd++) {
                const auto v = __builtin_amdgcn_permlane32_swap(m[odd][0], m[odd][1], false, false);
                t.q[WIDE ? odd : 0][WIDE ? d : 2 * odd + d] = v[0];
                t.q[WIDE ? 2 + odd : 1][WIDE ? d : 2 * odd + d] = v[1];
            }
        }
        const auto h = __builtin_amdgcn_permlane16_swap(t.h[0], t.h[1], false, false);
#pragma unroll
        for (int odd = 0; odd < 2; odd++) {
            const auto v = __builtin_amdgcn_permlane32_swap(h[odd], h[odd], false, false);
            hb[odd] = v[0];
            hb[2 + odd] = v[1];
        }
    }
}
// MFMA s of sub-step j takes eight columns per lane, of which lane c's are unit rows32_unit + c * rows32_lane of a row's 16.
template <int QT> constexpr int rows32_unit(int j, int s) {
    return Fmt<QT>::BITS == 8 ? 4 * j + s : QT == QT_NF4 ? 8 * (j / 2) + 4 * s + (j & 1) : 4 * j + 2 * s;
}
template <int QT> constexpr int rows32_lane() { return Fmt<QT>::BITS == 8 || QT == QT_NF4 ? 2 : 1; }

// MB: 32-row blocks of x per workgroup, 1 .. 5.  gridDim.y: the K splits, whose partial sums go to ws in register order.
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
    constexpr int BM = 32 * MB, XBYTES = BM * 256, PIECES = 2 * MB;      // 1 KB pieces of x (four rows) per wave and step
    constexpr int SUB = F::QK / 32, NS = 4 / SUB;            // sub-steps of 32 columns per scale; scales per step
    __shared__ __attribute__((aligned(1024))) uint8_t xs[2 * XBYTES];
    const int lane = threadIdx.x & 63, r = lane & 31, c = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

    const int grid_x = gridDim.x, splits = gridDim.y;
    // (one wait for all arguments: left alone the compiler loads each where it is first used, a scalar load's time apiece)
    asm volatile("" :: "s"(x), "s"(w), "s"(M), "s"(N), "s"(K), "s"(steps), "s"(ws), "s"(grid_x), "s"(splits));

    // Workgroups go to the XCDs in turn (id % 8): each XCD takes a run of the tiles, row tile by row tile within a column
    // tile, so that its L2 serves a column's weights to all their row tiles.
    // (With K splits what is dealt is tiles times splits, a tile's side by side: an eighth of the tiles in every split leaves some
    // XCDs with up to as many workgroups more as there are splits.  156 rows on [1281 x 6592] in asym_int4 took 1.23 times as
    // long, 136 on [1785 x 13248] in nf4 1.25, 85 random sizes 1.008 on average.)
    const int tiles_m = (M + BM - 1) / BM, tiles = tiles_m * ((N + RG_N - 1) / RG_N), xcd = blockIdx.x & 7;
    int tile = (tiles * xcd >> 3) + (int)(blockIdx.x >> 3), split = 0;       // (tiles below 2^27, see launch_gemm_rows)
    if (ws) {
        const int units = tiles * splits, first = units * xcd >> 3, count = (units * (xcd + 1) >> 3) - first;
        const int place = (int)((blockIdx.x >> 3) + blockIdx.y * (grid_x >> 3));
        if (place >= count) return;
        // Splits are of `steps` steps, the last one of what is left.  Where all workgroups beyond one per CU can be last splits, those
        // go out last (the CUs that two share would otherwise be the last to end: 56 rows on [8670 x 2176] in nf4, 272 workgroups
        // of 5, 5, 5 and 2 steps, 23.8 -> 19.0 us); elsewhere their order gains nothing (17 rows on [4685 x 13248] 1.06 times as long).
        const bool short_last = units > RG_CUS && units - RG_CUS <= tiles && splits * steps > (K + TILE_COLS - 1) / TILE_COLS;
        const int tile0 = tiles * xcd >> 3;                  // first / splits
        const int whole = short_last ? count - ((tiles * (xcd + 1) >> 3) - tile0) : count;
        const int at = short_last ? first - tile0 + place : first + place, per = short_last ? splits - 1 : splits;
        tile = place < whole ? at / per : tile0 + place - whole;
        split = place < whole ? at - tile * per : splits - 1;
    } else if (tile >= tiles * (xcd + 1) >> 3) return;       // whole workgroup leaves
    const int m0 = tile % tiles_m * BM, n0 = tile / tiles_m * RG_N + wave * 32;

    const int blocks = K / F::QK, G = (K + TILE_COLS - 1) / TILE_COLS;
    const int g0 = split * steps, g1 = g0 + steps < G ? g0 + steps : G;
    const int n = n0 + r;
    gbytes wr[2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int row = RowRegs32<QT>::SETS ? n0 + 16 * i + (lane & 15) : n;
        wr[i] = (gbytes)w + (int64_t)(row < N ? row : N - 1) * blocks * F::TS;
    }

    // x goes to LDS by itself: the 16 units (16 bytes) of a row's 128 columns in order, but for unit v of row m at v ^ m % 16,
    // so that the 32 rows that an MFMA operand takes a unit of spread over the banks.  A wave's piece i is rows 16i + 4 * wave
    // and the next three; rows past M are copies of the last one.
    const int xrow = 4 * wave + (lane >> 4), xunit = (lane & 15) ^ xrow;
    uint32_t xoff[PIECES];                                   // bytes from the tile's first row (K < 2^23)
#pragma unroll
    for (int i = 0; i < PIECES; i++) {
        const int m = i * 16 + xrow;
        xoff[i] = (uint32_t)(m0 + m < M ? m : M - 1 - m0) * (uint32_t)K * 2u;
    }
    const uint64_t xtile = (uint64_t)(uintptr_t)(x + (int64_t)m0 * K);
    const uint32_t xs_at = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)xs;
    auto dma_x = [&](int g, int buf, int p0, int p1) __attribute__((always_inline)) {
        // (past K: the group's first columns, times a scale of zero; from inline assembly, because the compiler would wait for
        // an LDS-DMA ahead of every later LDS access - a step ends by waiting for it)
        const uint32_t at = g * TILE_COLS + xunit * 8 < K ? (uint32_t)xunit * 16u : 0u;
        const uint64_t src = xtile + (uint64_t)g * (TILE_COLS * sizeof(AT));
        const uint32_t to = xs_at + buf + wave * 1024;
#pragma unroll
        for (int i = p0; i < p1; i++)
            asm volatile("s_add_u32 m0, %2, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                         :: "v"(xoff[i] + at), "s"(src), "s"(to), "n"(i * 4096) : "memory", "m0", "scc");
    };
    auto land = [&]() __attribute__((always_inline)) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    };

    f32x16 acc[MB];
    const f32x16 zero16 = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int mb = 0; mb < MB; mb++) acc[mb] = zero16;
    const V8 ones = ones8<AT>();
    const Op op;

    RowRegs32<QT> wc, wn;
    load_rows32<QT>(wr, g0, lane, blocks, wc);
    dma_x(g0, 0, 0, PIECES);
    land();
    // A step of 128 columns; the last one (more = false) loads nothing.  It stands apart from the loop: with a condition around
    // the loads the compiler merged the registers of this step's weights with the next one's where the ways met, and so
    // waited for the loads that it had just issued.
    int cur = 0;
    auto step = [&](int g, auto more_) __attribute__((always_inline)) {
        constexpr bool more = decltype(more_)::value;
        uint32_t hb[4];
        arrange_rows32<QT>(wc, hb);
        // MFMA o of the step: 32-row block mb, MFMA s of sub-step j, in the order of the units below
        constexpr int EARLY = QT == QT_FP8_E4M3 ? 0 : RowRegs32<QT>::NQ / 2;    // pieces of the weights loaded at the step's head
        constexpr int PER = 2 * SUB, OPS = NS * MB * PER, AHEAD = 3;
        const uint8_t *const base = xs + cur;
        const int at = r * 256 + ((c * rows32_lane<QT>()) ^ (r & 15)) * 16;
        auto read_x = [&](int o) __attribute__((always_inline)) {
            const int q = o / PER, t = o % PER, mb = q % MB, j = q / MB * SUB + t / 2;
            return *(const V8 *)(base + mb * 8192 + (at ^ (rows32_unit<QT>(j, t % 2) * 16)));
        };
        V8 a[AHEAD + 1], b[SUB == 1 ? 2 : 1][PER][PARTS];
        float d[2], e[2];                                    // of this scale and the next or the one before
        f32x16 p[2], sum[2];
        auto unpack = [&](int sc) __attribute__((always_inline)) {
#pragma unroll
            for (int jj = 0; jj < SUB; jj++) {
                const int j = sc * SUB + jj;
#pragma unroll
                for (int part = 0; part < PARTS; part++) {
                    V8 (&to)[PER][PARTS] = b[SUB == 1 ? sc & 1 : 0];
                    RowRegs<QT> t;
                    if constexpr (F::BITS == 8) {
                        t.q0 = wc.q[j];
                        to[2 * jj][part] = op.get(t, 0, part);
                        to[2 * jj + 1][part] = op.get(t, 1, part);
                    } else {
                        // bytes 0, 2, 1, 3: the unpacking then leaves low 0, 1, high 0, 1, low 2, 3, high 2, 3
                        V8 v[2];
#pragma unroll
                        for (int i = 0; i < 2; i++) {
                            const uint32_t dw = wc.q[j / 2][2 * (j & 1) + i];
                            t.q0[0] = __builtin_amdgcn_perm(dw, dw, 0x03010200u);
                            v[i] = op.get(t, 0, part);
                        }
                        to[2 * jj][part] = __builtin_shufflevector(v[0], v[1], 0, 1, 4, 5, 8, 9, 12, 13);
                        to[2 * jj + 1][part] = __builtin_shufflevector(v[0], v[1], 2, 3, 6, 7, 10, 11, 14, 15);
                    }
                }
            }
            float mn;
            hdr_to_scale<QT>(hb[sc * SUB], d[sc & 1], mn);
            e[sc & 1] = mn - OFFSET * d[sc & 1];
            d[sc & 1] = Op::scale(d[sc & 1]);
            asm volatile("" : "+v"(d[sc & 1]), "+v"(e[sc & 1]));      // (in fp32: not converted again in every FMA)
            if constexpr (!more) {                           // blocks past the end of the rows
                const bool past = g * NS + sc >= blocks;
                d[sc & 1] = past ? 0.0f : d[sc & 1];
                e[sc & 1] = past ? 0.0f : e[sc & 1];
            }
        };
#pragma unroll
        for (int o = 0; o < AHEAD && o < OPS; o++) a[o] = read_x(o);
        if constexpr (SUB == 1) unpack(0);
        // Unit q = (scale sc, 32-row block mb), in the order the hardware should issue them: an MFMA, the LDS read of x three
        // MFMAs ahead, a part of the scaling of the unit before, whose results have landed meanwhile, and so on; and the
        // unpacking of the next sub-step's weights (nf4 and fp8: of this scale's, ahead of its first unit).
        auto scale_some = [&](int q, int from, int to) __attribute__((always_inline)) {
            const int mb = q % MB, sc = q / MB;
#pragma unroll
            for (int i = from; i < to; i++) acc[mb][i] = Op::add(acc[mb][i], d[sc & 1], p[q & 1][i], e[sc & 1], sum[q & 1][i]);
        };
#pragma unroll
        for (int q = 0; q < NS * MB; q++) {
            const int sc = q / MB;
            if (SUB > 1 && q % MB == 0) {
                unpack(sc);
                __builtin_amdgcn_sched_barrier(0);
            }
            p[q & 1] = zero16;
            sum[q & 1] = zero16;
#pragma unroll
            for (int t = 0; t < PER; t++) {
                const int o = q * PER + t;
                if constexpr (more) {                        // the next step's x over the first half, its weights in the middle
#pragma unroll
                    for (int i = 0; i < PIECES; i++)
                        if (o == i * OPS / (2 * PIECES)) dma_x(g + 1, XBYTES - cur, i, i + 1);
                    if (EARLY && o == 0) load_rows32<QT>(wr, g + 1, lane, blocks, wn, 0, EARLY);
                    if (o == OPS / 2) load_rows32<QT>(wr, g + 1, lane, blocks, wn, EARLY);
                }
                const V8 v = a[o % (AHEAD + 1)];
                if constexpr (NEED_S) sum[q & 1] = mfma32(v, ones, sum[q & 1]);
#pragma unroll
                for (int part = 0; part < PARTS; part++) p[q & 1] = mfma32(v, b[SUB == 1 ? sc & 1 : 0][t][part], p[q & 1]);
                if (o + AHEAD < OPS) a[(o + AHEAD) % (AHEAD + 1)] = read_x(o + AHEAD);
                if (q > 0) scale_some(q - 1, t * 16 / PER, (t + 1) * 16 / PER);
                if (SUB == 1 && t == 1 && q % MB == MB / 2 && sc + 1 < NS) unpack(sc + 1);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        scale_some(NS * MB - 1, 0, 16);
        if constexpr (more) {
            land();
            wc = wn;
            cur = XBYTES - cur;
        }
    };
    int g = g0;
    for (; g + 1 < g1; g++) step(g, std::true_type{});
    step(g, std::false_type{});

    // C layout: lane = 32 * c + column (weight row), register 4q + i = row 8q + 4c + i of x
    if (ws) {
        f32x4 *part = (f32x4 *)ws + (((int64_t)split * tiles + tile) * RG_WAVES + wave) * (MB * 4 * 64) + lane;
#pragma unroll
        for (int mb = 0; mb < MB; mb++)
#pragma unroll
            for (int q = 0; q < 4; q++)
                part[(mb * 4 + q) * 64] = f32x4{acc[mb][4 * q], acc[mb][4 * q + 1], acc[mb][4 * q + 2], acc[mb][4 * q + 3]};
        return;
    }
    if (n >= N) return;
    const float bv = bias ? (float)bias[n] : 0.0f;
    uint64_t again[2] = {0, 0};                               // results that are not finite, see dot_fp32: of blocks 0 .. 3, and 4
#pragma unroll
    for (int mb = 0; mb < MB; mb++)
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int m = m0 + mb * 32 + i / 4 * 8 + c * 4 + i % 4;
            if (m < M) {
                y[(int64_t)m * N + n] = to_at<AT>(acc[mb][i] + bv);
                again[mb / 4] |= __builtin_isfinite(acc[mb][i]) ? 0ull : 1ull << (mb % 4 * 16 + i);
            }
        }
    while (again[0] | again[1]) {
        const int high = again[0] == 0, bit = __builtin_ctzll(high ? again[1] : again[0]);
        const int m = m0 + high * 128 + bit / 4 * 8 + c * 4 + bit % 4;
        y[(int64_t)m * N + n] = to_at<AT>(dot_fp32<QT, true>(x + (int64_t)m * K, w, n, K) + bv);
        if (high) again[1] &= again[1] - 1;
        else again[0] &= again[0] - 1;
    }
}

// Sums the splits and writes y, rounded once: one thread per four rows of one column.
template <int QT, typename AT, int MB>
__global__ __launch_bounds__(256) void gemm_rows_reduce_kernel(const f32x4 *__restrict__ ws, const AT *__restrict__ x,
                                                               const uint8_t *__restrict__ w, const AT *__restrict__ bias,
                                                               AT *__restrict__ y, int M, int N, int K, int tiles, int splits) {
    constexpr int PER_TILE = RG_WAVES * MB * 4 * 64;         // a multiple of 256
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int tiles_m = (M + 32 * MB - 1) / (32 * MB);
    const int tile = (int)(blockIdx.x / (PER_TILE / 256)), in = (int)(blockIdx.x % (PER_TILE / 256) * 256 + threadIdx.x);
    const int lane = in & 63, q = (in >> 6) & 3, mb = (in >> 8) % MB, wave = (in >> 8) / MB;
    const int m = tile % tiles_m * 32 * MB + mb * 32 + q * 8 + (lane >> 5) * 4;
    const int n = tile / tiles_m * RG_N + wave * 32 + (lane & 31);
    if (m >= M || n >= N) return;
    const f32x4 a = sum_splits(ws + t, (int64_t)tiles * PER_TILE, splits);
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
    double cost;                  // in steps of one row block, two workgroups per CU
};
// With row tiles of 32 * mb rows.  K splits: until the workgroups are about two per CU (the kernel's occupancy), of at least four
// steps each.  cost: a step reckons its weights as two row blocks, a workgroup that has a CU to itself takes 0.7 of the time, a split
// costs 2 and 5 per round of fp32 tiles.  (gemm_rows_us is a fit on top of it, to be made again when this changes.)
static RowsPlan rows_plan_of(int mb, int M, int N, int K, size_t ws_bytes) {
    RowsPlan p;
    p.mb = mb;
    p.tiles = ((M + 32 * mb - 1) / (32 * mb)) * ((N + RG_N - 1) / RG_N);
    const int G = (K + TILE_COLS - 1) / TILE_COLS;
    const size_t per_split = (size_t)p.tiles * 32 * mb * RG_N * sizeof(float);
    int s = 512 / p.tiles;
    s = s > G / 4 ? G / 4 : s;
    s = s > 16 ? 16 : s;
    while (s > 1 && (size_t)s * per_split > ws_bytes) s--;
    if (s < 1) s = 1;
    p.steps = (G + s - 1) / s;
    p.splits = (G + p.steps - 1) / p.steps;
    p.ws_bytes = p.splits > 1 ? p.splits * per_split : 0;
    const int64_t wgs = (int64_t)p.tiles * p.splits, per_cu = (wgs + 255) / 256;
    p.cost = p.steps * (mb + 2.0) * ((double)(per_cu / 2) + (per_cu % 2 ? 0.7 : 0.0)) + (p.splits > 1 ? 2.0 + 5.0 * (double)wgs * mb / 512 : 0.0);
    return p;
}
// Row tiles of 128 where they pad M by little more than 64 would, fewer for small batches and where 128 leave
// CUs idle, K too short to be split for them (200 rows on [1001 x 1088] 13.8 -> 12.1 us in sym_int4, 19.0 -> 15.4 in nf4; 128
// rows on [4001 x 2112] 17.4 -> 14.9 and 22.6 -> 19.8; with both forms at two workgroups per CU 64 rows lose, 256 rows on
// [30003 x 4096] 92 -> 124).  Tiles of 96 or 160 rows where their estimate is 8 % shorter: 80 rows on [9001 x 4096] in
// asym_int4 34.4 -> 28.3 us, 129 on [17563 x 3968] 78.5 -> 69.2 and in sym_int8 77.2 -> 53.5, 310 on [4677 x 4096] in sym_int4
// 37.8 -> 32.2, sym_int8 54.9 -> 37.0, nf4 47.3 -> 39.8; 1.025 times as fast over 330 random sizes, one of them slower by more than 4 % (143 rows on [5823 x 9216] in
// fp8_e4m3, 9 %).
static RowsPlan rows_plan_within(int qtype, int act_dtype, int M, int N, int K, size_t ws_bytes) {
    const int64_t pad64 = (M + 63) / 64 * 64, pad128 = (M + 127) / 128 * 128;
    RowsPlan p = rows_plan_of(M <= 32 ? 1 : M <= 64 || pad128 * 8 > pad64 * 9 ? 2 : 4, M, N, K, ws_bytes);
    const int G = (K + TILE_COLS - 1) / TILE_COLS;
    if (p.mb == 4 && (int64_t)p.tiles * (G / 4 > 1 ? G / 4 : 1) <= 256) return rows_plan_of(2, M, N, K, ws_bytes);
    if (M <= 32) return p;
    double best = 0.92 * p.cost;
    for (int mb = 3; mb <= 5; mb += 2) {
        if (mb == 5 && qtype == QT_NF4 && act_dtype == DT_BF16) continue;    // (nf4's three bf16 parts would spill)
        const RowsPlan other = rows_plan_of(mb, M, N, K, ws_bytes);
        if (other.cost < best) {
            p = other;
            best = other.cost;
        }
    }
    return p;
}
// A plan made again within its own bytes can lose, in 1 % of the sizes, to one whose splits the shortage of workspace takes away: that
// goes on until it comes out again, so that a workspace is sized for what is launched in it.  (The other way round, launching what
// was planned first, is 1.01 times as fast over 56 random sizes where both are split, 14 of them slower by more than 3 %, 0.83 at
// worst, and 0.79 over 34 where the second is not: 614 rows on [3879 x 960] in fp16 sym_int4 24.2 us against 14.7.)
static RowsPlan rows_plan(int qtype, int act_dtype, int M, int N, int K, size_t ws_bytes) {
    for (;;) {
        const RowsPlan p = rows_plan_within(qtype, act_dtype, M, N, K, ws_bytes);
        if (p.ws_bytes == ws_bytes) return p;
        ws_bytes = p.ws_bytes;
    }
}

// Sizes whose tiles 32-bit counts do not hold, or barely: neither planned nor launched.
static bool rows_too_many(int M, int N) {
    return M > 0x7fffff00 || N > 0x7fffff00 || (int64_t)((M + 15) / 16) * ((N + RG_N - 1) / RG_N) > 0x7ffffff;
}

size_t gemm_rows_workspace_bytes(int qtype, int act_dtype, int M, int N, int K, size_t max_bytes) {
    return rows_too_many(M, N) ? 0 : rows_plan(qtype, act_dtype, M, N, K, max_bytes).ws_bytes;
}

// What this kernel takes for M rows in microseconds, with all the workspace it asks for: fitted to 180 random sizes (M = 65 .. 512, N to
// 16384, K to 14000), 6 to 9 % rms.  0: not a size for it
double gemm_rows_us(int qtype, int act_dtype, int M, int N, int K) {
    if (rows_too_many(M, N)) return 0.0;
    const double cost = rows_plan(qtype, act_dtype, M, N, K, (size_t)256 << 20).cost;
    switch (qtype) {
    case QT_SYM_INT4: return 2.69 + 0.488 * cost;
    case QT_ASYM_INT4: return 1.26 + 0.737 * cost;
    case QT_SYM_INT8: return 2.17 + 0.605 * cost;
    case QT_NF4: return 1.57 + 0.760 * cost;
    default: return 1.65 + 0.472 * cost;
    }
}

template <int QT, typename AT, int MB>
static void launch_rows_m(const void *x, const void *w, const void *bias, void *y, int M, int N, int K, const RowsPlan &p, float *ws,
                          hipStream_t st) {
    if (p.splits == 1) ws = nullptr;
    hipLaunchKernelGGL((gemm_rows_kernel<QT, AT, MB>), dim3((p.tiles + 7) / 8 * 8, p.splits), dim3(256), 0, st, (const AT *)x,
                       (const uint8_t *)w, (const AT *)bias, (AT *)y, M, N, K, p.steps, ws);
    if (ws)
        hipLaunchKernelGGL((gemm_rows_reduce_kernel<QT, AT, MB>), dim3((unsigned)((int64_t)p.tiles * RG_WAVES * MB * 4 * 64 / 256)),
                           dim3(256), 0, st, (const f32x4 *)ws, (const AT *)x, (const uint8_t *)w, (const AT *)bias, (AT *)y, M, N, K,
                           p.tiles, p.splits);
}

template <int QT, typename AT>
static int launch_rows_t(const void *x, const void *w, const void *bias, void *y, int M, int N, int K, const RowsPlan &p, float *ws,
                         hipStream_t st) {
    if (p.mb == 1) launch_rows_m<QT, AT, 1>(x, w, bias, y, M, N, K, p, ws, st);
    else if (p.mb == 2) launch_rows_m<QT, AT, 2>(x, w, bias, y, M, N, K, p, ws, st);
    else if (p.mb == 3) launch_rows_m<QT, AT, 3>(x, w, bias, y, M, N, K, p, ws, st);
    else if (p.mb == 4) launch_rows_m<QT, AT, 4>(x, w, bias, y, M, N, K, p, ws, st);
    else if constexpr (QT != QT_NF4 || __is_same(AT, _Float16)) launch_rows_m<QT, AT, 5>(x, w, bias, y, M, N, K, p, ws, st);
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
    if (K >= (1 << 23))                                      // 32-bit offsets within a tile of x: the streaming kernel has 64
        return launch_gemv(x, w, bias, y, qtype, LAYOUT_GGML, act_dtype, M, N, K, 0, st);
    if (rows_too_many(M, N)) return -3;
    const RowsPlan p = rows_plan(qtype, act_dtype, M, N, K, workspace ? workspace_bytes : 0);
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
