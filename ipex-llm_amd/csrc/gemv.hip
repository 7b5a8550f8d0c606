// Decode-time product y[M,N] = x[M,K] * dequant(W)[N,K]^T for small M.
//
// Replaces xe_linear.forward_new at M = 1 and xe_batch.batch_forward at small M
// (python/llm/src/ipex_llm/transformers/low_bit_linear.py:657-668).
//
// gemv_mfma_kernel (tiled layout): HBM-bound streaming of the packed weights.
//   One workgroup owns one tile row (16 output columns) and its waves split
//   the 128-column tiles along K.  A lane's 16-byte load of a tile is already
//   its B operand for four v_mfma_f32_16x16x32 (one per 32-column sub-block);
//   codes are turned into exact small numbers in registers (never scaled in
//   half precision), the activations are the A operand (rows = batch index),
//   and the block scale is applied to the fp32 MFMA result.  M <= 16 costs the
//   same weight traffic as M = 1.  Algorithmic bytes per launch:
//   N*K*TS/QK (weights) + M*K*2 (x) + M*N*2 (y).
// The same kernel serves weights in the row-major (ggml) layout, whatever their shape (ROWS, lowbit_rows.h), and
// float32 activations (F32).
#include "lowbit_mfma.h"
#include "lowbit_rows.h"
#include "lowbit_unpack.h"

#include <type_traits>

namespace lowbit {

// ------------------------------------------------------------ MFMA GEMV

constexpr int GEMV_MAX_WAVES = 16;

constexpr int GEMV_LDS_X_BUDGET = 64 * 1024;

struct MoeId {
    int clamped;
    bool valid;
};
__device__ inline MoeId moe_id(const void *ids, bool ids64, int pair, int n_exp) {
    const int64_t e = ids64 ? ((const int64_t *)ids)[pair] : ((const int32_t *)ids)[pair];
    return {(int)(e < 0 ? 0 : e < n_exp ? e : n_exp - 1), e >= 0 && e < n_exp};
}

__device__ inline float load_route_w(const void *w, int dtype, int pair) {
    return dtype == DT_F32 ? ((const float *)w)[pair]
           : dtype == DT_F16 ? (float)((const _Float16 *)w)[pair] : (float)((const __bf16 *)w)[pair];
}

// One workgroup = one tile row (16 output columns).  Per round, wave w owns U consecutive
// tiles along K: it first issues every weight load of the round (so the whole slice is in
// flight at once), then copies its slice of x into a wave-private LDS region, then runs
// 4*U MFMAs whose A operand comes from LDS.  Rounds repeat until K is covered.
//
// DUAL: the fused gate/up projection of a gated MLP (xe_linear.mlp_forward_xpu,
// python/llm/src/ipex_llm/transformers/models/common.py:145-158): the workgroup walks the same
// tile row of two weights with one copy of x and writes act(x Wg^T) * (x Wu^T).
//
// MOE: the two launches of a fused mixture-of-experts decode step (xe_linear.moe_forward_vec,
// python/llm/src/ipex_llm/transformers/models/deepseek.py:290-315).  w / w2 are then tables of
// weight pointers in device memory and ids[j] names the expert of routing slot j, so that the host
// never has to read the routing result.
//   MOE == 1 (with DUAL): blockIdx.y = pair of token and slot; row blockIdx.y of y = act(x_t Wg[e]^T) * (x_t Wu[e]^T).
//   MOE == 2: blockIdx.y = token; x is its [slots, K / slots] part of the first launch's output, read as one long
//             vector; tile g of the K walk belongs to slot g / ge and is scaled by route_w[slot]:
//             y_t = sum_j route_w[j] * (x_j Wd[e_j]^T).
//   ids and route_w are read as the caller has them: 32- or 64-bit ids, weights of any float type.  A 64-bit id outside
//   [0, n_exp) takes its pair out of the sum; a 32-bit one stands for the nearest expert.
//
// F32 (lowbit_forward_f32): x, bias and y are float.  The MFMA operands are 16-bit, so AT is bf16 and each value of x
// becomes two on its way into LDS, hi = bf16(x) and lo = bf16(x - hi): 16 mantissa bits and fp32's exponent range.  Both
// go through the MFMA into the same fp32 accumulator.  (Splitting x in a kernel of its own, running its 2M rows as rows
// of a 16-bit product and adding the halves in a third kernel was 15.6 us of GPU time at 12 rows on [4096 x 4096] in
// sym_int4, two passes over the weights; this way it is one pass of 10.1 us.)
//
// ROWS: the weight is in the row-major layout and of any shape: N rows of which the last workgroup's may be fewer than
// 16, K any multiple of the block.  Loads and operand order as lowbit_rows.h says; everything else is the tiled
// kernel.  A row of a tile is 72 .. 136 contiguous bytes instead of a 1 KiB tile; a workgroup's waves take
// neighbouring columns, so lines are shared within the workgroup only.  (One wave per weight row and a scalar decode
// per weight, four rows of x a pass, took 74 us per pass for [32003 x 4096] in asym_int4: two at eight rows, which now take
// 29.8 us in bf16, 29.0 in fp16.)
template <int QT, typename AT, int MT, int U, int XN, bool DUAL, int MOE, int R, bool F32, bool ROWS>
__global__ __launch_bounds__(1024) void gemv_mfma_kernel(const AT *__restrict__ x, const uint8_t *__restrict__ w,
                                                         const uint8_t *__restrict__ w2, AT *__restrict__ y,
                                                         const AT *__restrict__ bias, int M, int N, int K, int act,
                                                         const void *__restrict__ ids, bool ids64,
                                                         const void *__restrict__ route_w, int route_dtype, int ge, int n_exp,
                                                         int slots) {
    using F = Fmt<QT>;
    using V8 = typename Vec8<AT>::type;
    using Op = Operand<QT, AT, F32, ROWS>;
    constexpr float OFFSET = Op::OFFSET;
    constexpr bool NEED_S = Op::NEED_S;
    // Row-major weights and the experts' pairs were products with decoded weights before they came here; tiled weights up to
    // eight rows never were.
    constexpr bool AGAIN = ROWS || MOE != 0;
    constexpr int SLICE = U * TILE_COLS;                    // columns of x per wave and round
    constexpr bool ZERO_X = XN == 1 || ROWS;                // how tiles past K are silenced (see the x loads)
    // With two planes of x that gains nothing and loses up to 15 % (5 rows on [2593 x 11648] in fp8_e4m3 13.8 -> 16.2 us), and the
    // forms left out with 16 bits lose up to 12 % at some sizes (3 rows on [32003 x 4096] in sym_int8 50 -> 52, 8 rows in asym_int4
    // 28.8 -> 30.1).  10000 random sizes: 1.008 times as fast with it as without, at worst 0.91 (asym_int4, 4 rows on
    // [3505 x 9792] 9.2 -> 10.1).
    constexpr bool ZERO_LATE = ROWS && XN > 1 && !F32 && !(MT == 2 && (QT == QT_FP8_E4M3 || QT == QT_ASYM_INT4)) &&
                               !(MT == 1 && XN == 4 && QT == QT_SYM_INT8);
    constexpr int XREGION = XN * 512 * (F32 ? 2 : 1);       // elements of AT in a wave's part of LDS

    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    // tile rows walked side by side with one copy of x: the same row of two weights (DUAL) or R
    // consecutive rows of one weight (worth it when M is large and N gives enough workgroups: at
    // M = 16 a workgroup otherwise pulls 3.5 bytes of x out of L2 per byte of weight)
    constexpr int NW = DUAL ? 2 : R;
    static_assert(!(DUAL && R != 1) && XN * 1024 >= NW * MT * 256, "bad GEMV shape parameters");
    static_assert(!ROWS || (!DUAL && MOE == 0), "row-major weights: the plain product only");
    const Op op;
    constexpr bool NF4_IN_LDS = QT == QT_NF4 && MT == 1 && Op::PARTS == 1;     // (see Unpack<QT_NF4>)
    __shared__ AT lut_lds[16];
    if constexpr (NF4_IN_LDS) {
        if (threadIdx.x < 16) lut_lds[threadIdx.x] = to_at<AT>(NF4_CODEBOOK[threadIdx.x]);
        __syncthreads();
    }

    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, W = blockDim.x >> 6;
    const int G = ROWS ? (K + TILE_COLS - 1) / TILE_COLS : K / TILE_COLS;
    const int r = lane & 15, c = lane >> 4;
    // A rows: row r carries batch index (r/4)*MT + r%4 when r%4 < MT, so that the C registers
    // i < MT of lane group g hold batch indices g*MT + i and nothing else has to be scaled.
    // Rows with r%4 >= MT (and batch indices >= M) only feed C rows that are never read, so
    // they may hold anything: they re-read a valid row, which LDS serves as a broadcast.
    int m_of_r = (r >> 2) * MT + ((r & 3) < MT ? (r & 3) : MT - 1);
    m_of_r = m_of_r < M ? m_of_r : M - 1;
    gbytes wrow = nullptr, wrow2 = nullptr;
    gbytes wr[ROWS ? R : 1];                                // ROWS: this lane's row of each tile row
    const int blocks = K / F::QK;
    if constexpr (ROWS) {
#pragma unroll
        for (int wi = 0; wi < R; wi++) {
            const int64_t n = ((int64_t)blockIdx.x * R + wi) * TILE_ROWS + r;
            wr[wi] = (gbytes)w + (n < N ? n : N - 1) * (int64_t)blocks * F::TS;
        }
    } else if constexpr (MOE == 0) {
        wrow = (gbytes)w + (int64_t)blockIdx.x * R * G * F::TILE_BYTES;
        if constexpr (DUAL) wrow2 = (gbytes)w2 + (int64_t)blockIdx.x * G * F::TILE_BYTES;
    } else if constexpr (MOE == 1) {
        // ids come from device memory: clamp, so that a bad id cannot send a load astray
        const int e = moe_id(ids, ids64, blockIdx.y, n_exp).clamped;
        wrow = (gbytes)((const uint8_t *const *)w)[e] + (int64_t)blockIdx.x * G * F::TILE_BYTES;
        wrow2 = (gbytes)((const uint8_t *const *)w2)[e] + (int64_t)blockIdx.x * G * F::TILE_BYTES;
        x += (int64_t)(blockIdx.y / slots) * K;
        y += (int64_t)blockIdx.y * N;
    } else {
        x += (int64_t)blockIdx.y * K;
        y += (int64_t)blockIdx.y * N;
    }
    // MOE == 2: tile g -> slot g / ge; its weight row starts at table[ids[slot]] + blockIdx.x * ge tiles.  Lane j looks slot
    // j up once (at most 64 slots), a tile then asks that lane: per tile, the chain id -> pointer -> weight and the
    // branches on the types of ids and weights cost 3 us of 6 (60 experts of [1408 x 2048], four slots).
    uint64_t slot_w = 0;
    float slot_rw = 0.0f;
    if constexpr (MOE == 2) {
        const int pair = blockIdx.y * slots + (lane < slots ? lane : 0);
        const MoeId id = moe_id(ids, ids64, pair, n_exp);
        slot_w = (uint64_t)((const uint8_t *const *)w)[id.clamped];
        slot_rw = load_route_w(route_w, route_dtype, pair);
        if (ids64 && !id.valid) slot_rw = 0.0f;
    }
    auto moe_tile = [&](int g, float &rw) -> gbytes {
        const int slot = __builtin_amdgcn_readfirstlane(g / ge);
        rw = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, slot_rw), slot));
        const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)slot_w, slot);
        const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(slot_w >> 32), slot);
        return (gbytes)((uint64_t)lo | ((uint64_t)hi << 32)) + ((int64_t)blockIdx.x * ge + (g - slot * ge)) * F::TILE_BYTES;
    };
    AT *xs = (AT *)smem + (int64_t)wave * XREGION;          // [XN*64/(SLICE/8)][SLICE], private to this wave
    const AT *xa = xs + m_of_r * SLICE + 8 * c;

    float acc[NW * MT];
#pragma unroll
    for (int i = 0; i < NW * MT; i++) acc[i] = 0.0f;
    const V8 ones = ones8<AT>();
    const f32x4 zero4 = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int g0 = 0; g0 < G; g0 += W * U) {
        const int gw = g0 + wave * U;
        // Straight-line loads (addresses clamped instead of branches, so that the compiler can
        // count outstanding loads): x first - it comes from L2 and is needed before any MFMA -
        // then every weight tile of the round.  Loads return in order, so the LDS copy of x
        // waits for the x loads only and each tile is consumed as soon as it lands while the
        // later ones are still in flight.  XN = 16-byte chunks of x per lane (>= M*U/4).
        u32x4 xv[F32 ? 2 * XN : XN];
#pragma unroll
        for (int i = 0; i < XN; i++) {
            const int idx = i * 64 + lane;
            int m = idx / (SLICE / 8);
            const int u = idx % (SLICE / 8);
            int col = gw * TILE_COLS + u * 8;
            m = m < M ? m : M - 1;
            // Columns past K (tiles of the last round that a wave has no work for).  With one chunk of x per lane x
            // reads as zero there - the weights of the tile that stands in, the row's last, are finite - which is
            // one select per round where zeroing the scales is one per sub-block (M = 1: [11008 x 4096] 6.23 ->
            // 6.15 us, [28672 x 8192] 24.8 -> 23.8); with more chunks per lane the same change cost 5-20 %, and
            // those shapes zero the scales (below).
            // Row-major weights with more chunks select where x goes to LDS (ZERO_LATE): here the select waits for x in front of
            // the loads of the weights (8 rows on [32003 x 4096] in sym_int8 56.0 -> 53.2 us).  With one chunk the compiler has
            // moved it behind them by itself.
            const bool past = col >= K;
            col = past ? K - 8 : col;
            if constexpr (F32) {
                const u32x4 *xp = (const u32x4 *)((const float *)x + (int64_t)m * K + col);
                xv[2 * i] = xp[0];
                xv[2 * i + 1] = xp[1];
                if constexpr (ZERO_X && !ZERO_LATE) {
                    xv[2 * i] = past ? u32x4{0u, 0u, 0u, 0u} : xv[2 * i];
                    xv[2 * i + 1] = past ? u32x4{0u, 0u, 0u, 0u} : xv[2 * i + 1];
                }
            } else {
                xv[i] = *(const u32x4 *)(x + (int64_t)m * K + col);
                if constexpr (ZERO_X && !ZERO_LATE) xv[i] = past ? u32x4{0u, 0u, 0u, 0u} : xv[i];
            }
        }
        __builtin_amdgcn_sched_barrier(0);                  // keep the x loads ahead of the weight loads
        typename std::conditional<ROWS, RowRegs<QT>, TileRegs<QT>>::type tr[NW * U];
        float rw[U];
        if constexpr (ROWS) {
#pragma unroll
            for (int wi = 0; wi < R; wi++)
#pragma unroll
                for (int t = 0; t < U; t++) load_rows<QT>(wr[wi], gw + t < G ? gw + t : G - 1, c, blocks, tr[wi * U + t]);
        } else {
#pragma unroll
            for (int t = 0; t < U; t++) {
                const int g = gw + t < G ? gw + t : G - 1;
                rw[t] = 1.0f;
                if constexpr (MOE == 2) load_tile<QT, true>(moe_tile(g, rw[t]), lane, r, tr[t]);
                else load_tile<QT, true>(wrow + (int64_t)g * F::TILE_BYTES, lane, r, tr[t]);
            }
            if constexpr (DUAL) {
#pragma unroll
                for (int t = 0; t < U; t++) {
                    const int g = gw + t;
                    load_tile<QT, true>(wrow2 + (int64_t)(g < G ? g : G - 1) * F::TILE_BYTES, lane, r, tr[U + t]);
                }
            }
#pragma unroll
            for (int wi = 1; wi < R; wi++)
#pragma unroll
                for (int t = 0; t < U; t++) {
                    const int g = gw + t < G ? gw + t : G - 1;
                    load_tile<QT, true>(wrow + ((int64_t)wi * G + g) * F::TILE_BYTES, lane, r, tr[wi * U + t]);
                }
        }

        __builtin_amdgcn_sched_barrier(0);
        // The LDS region is private to the wave and LDS operations of a wave execute in order:
        // a wavefront-scope fence (no hardware wait) is all the synchronization it needs.
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int i = 0; i < XN; i++) {
            const int at = i * 64 + lane;
            auto put = [&](AT *plane, const u32x4 &v) __attribute__((always_inline)) {
                if constexpr (ROWS) store_x_rows<QT>((uint8_t *)(plane + at / (SLICE / 8) * SLICE), at % (SLICE / 8), v);
                else *(u32x4 *)(plane + at * 8) = v;
            };
            if constexpr (ZERO_LATE) {
                const bool past = (int)(gw * TILE_COLS + at % (SLICE / 8) * 8) >= K;
                xv[i] = past ? u32x4{0u, 0u, 0u, 0u} : xv[i];
            }
            if constexpr (F32) {
                u32x4 hi, lo;
                split_f32(xv[2 * i], xv[2 * i + 1], hi, lo);
                put(xs, hi);
                put(xs + XN * 512, lo);
            } else {
                put(xs, xv[i]);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();

#pragma unroll
        for (int wi = 0; wi < NW; wi++)
#pragma unroll
            for (int t = 0; t < U; t++) {
                auto &tl = tr[wi * U + t];
                uint32_t hb[4];
                if constexpr (ROWS) arrange_rows<QT>(tl, hb);
                const bool live = ZERO_X || gw + t < G;
                V8 a[4], al[4];
#pragma unroll
                for (int j = 0; j < 4; j++) a[j] = *(const V8 *)(xa + (t * 4 + j) * 32);
                if constexpr (F32) {
#pragma unroll
                    for (int j = 0; j < 4; j++) al[j] = *(const V8 *)(xa + XN * 512 + (t * 4 + j) * 32);
                }
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    V8 b[Op::PARTS];
#pragma unroll
                    for (int part = 0; part < Op::PARTS; part++) {
                        if constexpr (NF4_IN_LDS) b[part] = Unpack<QT, AT>::run_lds(tl.q0[j], lut_lds);
                        else b[part] = op.get(tl, j, part);
                    }
                    float d, mn;
                    if constexpr (ROWS) hdr_to_scale<QT>(hb[j], d, mn);
                    else tile_scale<QT>(tl, j, d, mn);
                    if constexpr (MOE == 2) {
                        d *= rw[t];
                        mn *= rw[t];
                    }
                    if constexpr (!ZERO_X) {
                        d = live ? d : 0.0f;
                        mn = live ? mn : 0.0f;
                    }
                    const f32x4 p = Op::product(a[j], al[j], b);
                    f32x4 s = zero4;
                    if constexpr (NEED_S) {
                        s = mfma16(a[j], ones, zero4);
                        if constexpr (F32) s = mfma16(al[j], ones, s);
                    }
                    const float e = mn - OFFSET * d;
                    d = Op::scale(d);
#pragma unroll
                    for (int i = 0; i < MT; i++) acc[wi * MT + i] = Op::add(acc[wi * MT + i], d, p[i], e, s[i]);
                }
            }
    }

    // sum the K-slices of the waves; wave 0 writes.  C layout: lane = 16*grp + col, register i = row 4*grp + i.
    // The partial sums go to the start of each wave's own x region, which is dead by now.
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    float *red = (float *)smem;
    constexpr int RS = XREGION / 2;                         // floats per wave region
#pragma unroll
    for (int i = 0; i < NW * MT; i++) red[wave * RS + i * 64 + lane] = acc[i];
    __syncthreads();
    // wave v sums and writes tile row v of the R rows (DUAL: wave 0 combines both weights)
    if (wave < (DUAL ? 1 : R)) {
        const int grp = lane >> 4, col = lane & 15;
        const int64_t n = ((int64_t)blockIdx.x * R + wave) * 16 + col;
        auto store = [&](int m, float s, float up) __attribute__((always_inline)) {
            if constexpr (DUAL) s = gate_act(s, act) * up;
            if constexpr (F32) {
                ((float *)y)[(int64_t)m * N + n] = bias ? s + ((const float *)bias)[n] : s;
            } else {
                if constexpr (!DUAL && MOE == 0) s += bias ? (float)bias[n] : 0.0f;
                y[(int64_t)m * N + n] = to_at<AT>(s);
            }
        };
        uint32_t again = 0;                                 // AGAIN: results that are not finite, see dot_fp32
#pragma unroll
        for (int i = 0; i < MT; i++) {
            float s = 0.0f, up = 0.0f;
            for (int ww = 0; ww < W; ww++) s += red[ww * RS + (wave * MT + i) * 64 + lane];
            if constexpr (DUAL) {
                for (int ww = 0; ww < W; ww++) up += red[ww * RS + (MT + i) * 64 + lane];
            }
            const int m = grp * MT + i;
            if (m >= M || (ROWS && n >= N)) continue;
            store(m, s, up);
            if constexpr (AGAIN) again |= __builtin_isfinite(s) && __builtin_isfinite(up) ? 0u : 1u << i;
        }
        for (; AGAIN && again; again &= again - 1) {
            const int m = grp * MT + __builtin_ctz(again);
            using ET = typename std::conditional<F32, float, AT>::type;
            const ET *row = (const ET *)x + (int64_t)m * K;
            if constexpr (MOE == 0) {
                store(m, dot_fp32<QT, ROWS>(row, w, n, K), 0.0f);
            } else if constexpr (MOE == 1) {
                const int e = moe_id(ids, ids64, blockIdx.y, n_exp).clamped;
                store(m, dot_fp32<QT, false>(row, ((const uint8_t *const *)w)[e], n, K),
                      dot_fp32<QT, false>(row, ((const uint8_t *const *)w2)[e], n, K));
            } else {
                float s = 0.0f;
                for (int slot = 0; slot < slots; slot++) {
                    const int pair = blockIdx.y * slots + slot;
                    const MoeId id = moe_id(ids, ids64, pair, n_exp);
                    if (ids64 && !id.valid) continue;
                    s += load_route_w(route_w, route_dtype, pair) *
                         dot_fp32<QT, false>(row + (int64_t)slot * ge * TILE_COLS, ((const uint8_t *const *)w)[id.clamped], n,
                                             (int64_t)ge * TILE_COLS);
                }
                store(m, s, 0.0f);
            }
        }
    }
}

// -------------------------------------------------------------- launch

struct GemvExtra {                                          // what the fused forms take besides
    const uint8_t *w2 = nullptr;
    int act = 0;
    const void *ids = nullptr;
    bool ids64 = false;
    const void *route_w = nullptr;
    int route_dtype = DT_F32;
    int ge = 0, slots = 1, n_exp = 1, tokens = 1;
};

template <int QT, typename AT, int MT, int U, int XN, bool DUAL = false, int MOE = 0, int R = 1, bool F32 = false, bool ROWS = false>
static void launch_mfma(const AT *x, const uint8_t *w, const AT *bias, AT *y, int M, int N, int K, int waves, hipStream_t st,
                        const GemvExtra &e = {}) {
    constexpr int XBYTES = XN * 1024 * (F32 ? 2 : 1);       // of x in LDS per wave
    const int G = (K + TILE_COLS - 1) / TILE_COLS;
    // waves: enough that one round covers K, within the block size limit and the LDS budget for x
    int wv = (G + U - 1) / U;
    const int lds_cap = GEMV_LDS_X_BUDGET / XBYTES;
    if (wv > lds_cap) wv = lds_cap;
    if (wv > GEMV_MAX_WAVES) wv = GEMV_MAX_WAVES;
    if (waves > 0 && waves < wv) wv = waves;
    if (wv < R) wv = R;                                     // (wave v writes tile row v)
    if (wv < 1) wv = 1;
    hipLaunchKernelGGL((gemv_mfma_kernel<QT, AT, MT, U, XN, DUAL, MOE, R, F32, ROWS>),
                       dim3((N + TILE_ROWS * R - 1) / (TILE_ROWS * R), MOE == 1 ? e.tokens * e.slots : MOE == 2 ? e.tokens : 1), dim3(64 * wv), (size_t)wv * XBYTES, st,
                       x, w, e.w2, y, bias, M, N, K, e.act, e.ids, e.ids64, e.route_w,
                       e.route_dtype, e.ge, e.n_exp, e.slots);
}

template <int QT, typename AT, bool F32, bool ROWS>
static int launch_gemv_t(const void *x, const void *w, const void *bias, void *y, int M, int N, int K, int waves, hipStream_t st) {
    using ET = typename std::conditional<F32, float, AT>::type;
    const int tile_rows = (N + TILE_ROWS - 1) / TILE_ROWS;
    // tile rows may share x in groups of R when R divides them; a row-major weight's last group may reach past its end
    auto shares = [&](int R) { return ROWS || tile_rows % R == 0; };
    const uint8_t *wp = (const uint8_t *)w;
    const AT *b = (const AT *)bias;
    for (int m0 = 0; m0 < M; m0 += 16) {
        const int mc = (M - m0) < 16 ? (M - m0) : 16;
        const AT *xp = (const AT *)((const ET *)x + (int64_t)m0 * K);
        AT *yp = (AT *)((ET *)y + (int64_t)m0 * N);
        // Tiles per wave and round (U), measured on MI355X: 4 when K fits one round of 8 waves and
        // there are many tile rows to spread over the CUs, else 2 with up to 16 waves and as many
        // rounds as K needs.  XN = chunks of eight columns of x per lane = ceil(M * U / 4).
        const bool u4 = !F32 && (K + TILE_COLS - 1) / TILE_COLS <= 32 && N >= 8192;
        if (mc <= 4) {
            if constexpr (!F32) {
                if (u4) {
                    if (mc == 1) launch_mfma<QT, AT, 1, 4, 1, false, 0, 1, F32, ROWS>(xp, wp, b, yp, mc, N, K, waves, st);
                    else if (mc == 2) launch_mfma<QT, AT, 1, 4, 2, false, 0, 1, F32, ROWS>(xp, wp, b, yp, mc, N, K, waves, st);
                    else launch_mfma<QT, AT, 1, 4, 4, false, 0, 1, F32, ROWS>(xp, wp, b, yp, mc, N, K, waves, st);
                    continue;
                }
            }
            if (mc <= 2) launch_mfma<QT, AT, 1, 2, 1, false, 0, 1, F32, ROWS>(xp, wp, b, yp, mc, N, K, waves, st);
            else launch_mfma<QT, AT, 1, 2, 2, false, 0, 1, F32, ROWS>(xp, wp, b, yp, mc, N, K, waves, st);
        }
        // 5 .. 8 rows: one tile per wave and round with up to 16 waves keeps the x slice of a wave (and with
        // it the workgroup's LDS footprint) small; two tile rows share x where N leaves enough workgroups
        // (measured on MI355X, sym_int4: 5-7 % on the Llama-2-7B shapes, 15-20 % on [28672 x 8192] and
        // [8192 x 28672] against four tiles per wave)
        else if (mc <= 8 && shares(2) && N >= 8192)
            launch_mfma<QT, AT, 2, 1, 2, false, 0, 2, F32, ROWS>(xp, wp, b, yp, mc, N, K, waves, st);
        else if (mc <= 8) launch_mfma<QT, AT, 2, 1, 2, false, 0, 1, F32, ROWS>(xp, wp, b, yp, mc, N, K, waves, st);
        else if constexpr (F32) return -7;                  // (9 rows and more: gemv_wide.hip)
        // 9 .. 16 rows of x: share x between 4 or 2 tile rows where N still gives enough workgroups
        // (measured on MI355X: +25 .. 70 % on [28672 x 8192], +8 .. 24 % on [8192 x 8192])
        else if (shares(4) && N >= 16384)
            launch_mfma<QT, AT, 4, 1, 4, false, 0, 4, F32, ROWS>(xp, wp, b, yp, mc, N, K, waves, st);
        else if (shares(2) && N >= 8192 && K >= 8192)
            launch_mfma<QT, AT, 4, 1, 4, false, 0, 2, F32, ROWS>(xp, wp, b, yp, mc, N, K, waves, st);
        else if (shares(2) && N >= 8192)
            launch_mfma<QT, AT, 4, 2, 8, false, 0, 2, F32, ROWS>(xp, wp, b, yp, mc, N, K, waves, st);
        else launch_mfma<QT, AT, 4, 2, 8, false, 0, 1, F32, ROWS>(xp, wp, b, yp, mc, N, K, waves, st);
    }
    return 0;
}

template <int QT, bool ROWS>
static int launch_gemv_dt(const void *x, const void *w, const void *bias, void *y, int dt, int M, int N, int K, int waves,
                          hipStream_t st) {
    if (dt == DT_F16) return launch_gemv_t<QT, _Float16, false, ROWS>(x, w, bias, y, M, N, K, waves, st);
    if (dt == DT_BF16) return launch_gemv_t<QT, __bf16, false, ROWS>(x, w, bias, y, M, N, K, waves, st);
    if (dt == DT_F32) return launch_gemv_t<QT, __bf16, true, ROWS>(x, w, bias, y, M, N, K, waves, st);
    return -4;
}

template <int QT>
static int launch_gemv_q(const void *x, const void *w, const void *bias, void *y, int layout, int dt, int M, int N, int K, int waves,
                         hipStream_t st) {
    if (layout == LAYOUT_TILED) {
        if (N % TILE_ROWS || K % TILE_COLS) return -5;
        return launch_gemv_dt<QT, false>(x, w, bias, y, dt, M, N, K, waves, st);
    }
    return launch_gemv_dt<QT, true>(x, w, bias, y, dt, M, N, K, waves, st);
}

template <int QT, typename AT>
static int launch_mlp_t(const void *x, const void *wg, const void *wu, void *y, int M, int N, int K, int act,
                        hipStream_t st) {
    // Two tiles of each weight per wave and round, at most 8 waves: the registers of four tiles in flight
    // keep the kernel below 80 vector registers, so that a CU holds three workgroups and the 688 workgroups
    // of a [11008 x 4096] pair all run side by side.  With four tiles of each weight the kernel takes 120
    // registers and a third of the workgroups has to wait for a free slot.
    const uint8_t *g = (const uint8_t *)wg;
    GemvExtra e;
    e.w2 = (const uint8_t *)wu;
    e.act = act;
    const AT *xp = (const AT *)x;
    AT *yp = (AT *)y;
    if (M <= 2) launch_mfma<QT, AT, 1, 2, 1, true>(xp, g, nullptr, yp, M, N, K, 8, st, e);
    else if (M <= 4) launch_mfma<QT, AT, 1, 2, 2, true>(xp, g, nullptr, yp, M, N, K, 8, st, e);
    // 5 .. 8 rows: one tile of each weight per wave and round with up to 16 waves, as the plain product's
    // kernels that share x between two tile rows
    else if (M <= 8) launch_mfma<QT, AT, 2, 1, 2, true>(xp, g, nullptr, yp, M, N, K, 0, st, e);
    else return -7;
    return 0;
}

template <int QT>
static int launch_mlp_q(const void *x, const void *wg, const void *wu, void *y, int dt, int M, int N, int K, int act,
                        hipStream_t st) {
    if (dt == DT_F16) return launch_mlp_t<QT, _Float16>(x, wg, wu, y, M, N, K, act, st);
    if (dt == DT_BF16) return launch_mlp_t<QT, __bf16>(x, wg, wu, y, M, N, K, act, st);
    return -4;
}

// y[M, N] = act(x Wg^T) * (x Wu^T) for up to 8 rows, both weights tiled [N, K]
int launch_mlp_gemv(const void *x, const void *wg, const void *wu, void *y, int qtype, int act_dtype, int M, int N,
                    int K, int act, hipStream_t st) {
    if (M == 0 || N == 0) return 0;
    switch (qtype) {
    case QT_SYM_INT4: return launch_mlp_q<QT_SYM_INT4>(x, wg, wu, y, act_dtype, M, N, K, act, st);
    case QT_ASYM_INT4: return launch_mlp_q<QT_ASYM_INT4>(x, wg, wu, y, act_dtype, M, N, K, act, st);
    case QT_SYM_INT8: return launch_mlp_q<QT_SYM_INT8>(x, wg, wu, y, act_dtype, M, N, K, act, st);
    case QT_NF4: return launch_mlp_q<QT_NF4>(x, wg, wu, y, act_dtype, M, N, K, act, st);
    case QT_FP8_E4M3: return launch_mlp_q<QT_FP8_E4M3>(x, wg, wu, y, act_dtype, M, N, K, act, st);
    default: return -2;
    }
}

// h[pair, inter] = act(x_t Wg[e]^T) * (x_t Wu[e]^T) for every pair of token and slot, then
// y[t, hidden] = sum_j route_w[t, j] * (h[t, j] Wd[e_j]^T).  e holds what both launches share.
template <int QT, typename AT>
static int launch_moe_t(const void *x, const void *gates, const void *downs, void *h, void *y, int hidden, int inter, const GemvExtra &e,
                        hipStream_t st) {
    launch_mfma<QT, AT, 1, 4, 1, true, 1>((const AT *)x, (const uint8_t *)gates, nullptr, (AT *)h, 1, inter, hidden, 0, st, e);
    launch_mfma<QT, AT, 1, 4, 1, false, 2>((const AT *)h, (const uint8_t *)downs, nullptr, (AT *)y, 1, hidden, e.slots * inter, 0, st, e);
    return 0;
}

template <int QT>
static int launch_moe_q(const void *x, const void *gates, const void *downs, void *h, void *y, int dt, int hidden, int inter,
                        const GemvExtra &e, hipStream_t st) {
    if (dt == DT_F16) return launch_moe_t<QT, _Float16>(x, gates, downs, h, y, hidden, inter, e, st);
    if (dt == DT_BF16) return launch_moe_t<QT, __bf16>(x, gates, downs, h, y, hidden, inter, e, st);
    return -4;
}

int launch_moe_gemv(const void *x, const void *ids, bool ids64, const void *route_w, int route_dtype, int tokens, int top_k,
                    int n_exp, const void *gates, const void *ups, const void *downs, void *h, void *y, int qtype, int act_dtype,
                    int hidden, int inter, int act, hipStream_t st) {
    GemvExtra e;
    e.w2 = (const uint8_t *)ups;
    e.act = act;
    e.ids = ids;
    e.ids64 = ids64;
    e.route_w = route_w;
    e.route_dtype = route_dtype;
    e.ge = inter / TILE_COLS;
    e.slots = top_k;
    e.n_exp = n_exp;
    e.tokens = tokens;
    switch (qtype) {
    case QT_SYM_INT4: return launch_moe_q<QT_SYM_INT4>(x, gates, downs, h, y, act_dtype, hidden, inter, e, st);
    case QT_ASYM_INT4: return launch_moe_q<QT_ASYM_INT4>(x, gates, downs, h, y, act_dtype, hidden, inter, e, st);
    case QT_SYM_INT8: return launch_moe_q<QT_SYM_INT8>(x, gates, downs, h, y, act_dtype, hidden, inter, e, st);
    case QT_NF4: return launch_moe_q<QT_NF4>(x, gates, downs, h, y, act_dtype, hidden, inter, e, st);
    case QT_FP8_E4M3: return launch_moe_q<QT_FP8_E4M3>(x, gates, downs, h, y, act_dtype, hidden, inter, e, st);
    default: return -2;
    }
}

// y[M, N] = x[M, K] * dequant(w)^T (+ bias, which may be null) in passes of 16 rows; x, bias and y of act_dtype, which may
// be DT_F32 (see F32)
int launch_gemv(const void *x, const void *w, const void *bias, void *y, int qtype, int layout, int act_dtype, int M, int N,
                int K, int waves, hipStream_t st) {
    if (M == 0 || N == 0) return 0;
    switch (qtype) {
    case QT_SYM_INT4: return launch_gemv_q<QT_SYM_INT4>(x, w, bias, y, layout, act_dtype, M, N, K, waves, st);
    case QT_ASYM_INT4: return launch_gemv_q<QT_ASYM_INT4>(x, w, bias, y, layout, act_dtype, M, N, K, waves, st);
    case QT_SYM_INT8: return launch_gemv_q<QT_SYM_INT8>(x, w, bias, y, layout, act_dtype, M, N, K, waves, st);
    case QT_NF4: return launch_gemv_q<QT_NF4>(x, w, bias, y, layout, act_dtype, M, N, K, waves, st);
    case QT_FP8_E4M3: return launch_gemv_q<QT_FP8_E4M3>(x, w, bias, y, layout, act_dtype, M, N, K, waves, st);
    default: return -2;
    }
}

}  // namespace lowbit
