// Weights in the row-major (ggml) layout as operands of v_mfma_f32_16x16x32: what the streaming kernel and the one-pass
// kernel share (larger products: gemm_rows.hip, in 32 x 32 tiles).
//
// Both take 16 weight rows by 128 columns at a time, lane l = 16*c + r standing for row r.  A lane loads 16 bytes of
// codes per load (8-bit formats: twice) at the 2-byte alignment that the blocks have, and the header in front:
//   sym_int4, asym_int4, sym_int8   lane c takes block c of the four 32-weight blocks
//   nf4                             lane c takes half c % 2 of block c / 2 (64 weights, 32 bytes)
//   fp8_e4m3                        lane c takes bytes 32c .. 32c+31 of the one 128-weight block
// An MFMA has to stay within one block, whose scale is applied to its fp32 result.  So for all but fp8 the four dwords
// of the four lanes of a row are transposed (two rounds of v_permlane32_swap / v_permlane16_swap): register j then holds
// dword c of what lane j had loaded, and MFMA step j covers that block (half block) alone.  Which columns a lane holds
// is the format's business (low nibbles are the first half of a block); a product does not mind the order of the
// columns as long as x has the same one, so x is permuted on its way into LDS (store_x_rows) and stays a 16-byte read:
//   4-bit   step j of lane c: codes 4c .. 4c+3 in the low nibbles (columns 4c+i) and in the high ones (columns 16+4c+i;
//           nf4: 32+4c+i), in the order the unpacking leaves them: lo0, lo2, hi0, hi2, lo1, lo3, hi1, hi3
//   int8    step j of lane c: columns 4c .. 4c+3, 16+4c .. 16+4c+3 of block j
//   fp8     step j of lane c: columns 32c+8j .. 32c+8j+7
#pragma once
#include "lowbit_mfma.h"

namespace lowbit {

typedef uint32_t u32x4_a2 __attribute__((ext_vector_type(4), aligned(2)));
typedef uint32_t u32_a2 __attribute__((aligned(2)));

// The header of the block that lane row j loaded, in all lanes, for j = 0 .. 3
__device__ inline void spread_rows(uint32_t h, uint32_t (&hb)[4]) {
    const auto p = __builtin_amdgcn_permlane32_swap(h, h, false, false);          // rows 0 1 0 1 / 2 3 2 3
    const auto a = __builtin_amdgcn_permlane16_swap(p[0], p[0], false, false);
    const auto b = __builtin_amdgcn_permlane16_swap(p[1], p[1], false, false);
    hb[0] = a[0]; hb[1] = a[1]; hb[2] = b[0]; hb[3] = b[1];
}
// v[j] in lane row c  ->  v[c] of lane row j
__device__ inline u32x4 transpose_rows(const u32x4 &v) {
    const auto p = __builtin_amdgcn_permlane32_swap(v[0], v[2], false, false);
    const auto q = __builtin_amdgcn_permlane32_swap(v[1], v[3], false, false);
    const auto a = __builtin_amdgcn_permlane16_swap(p[0], q[0], false, false);
    const auto b = __builtin_amdgcn_permlane16_swap(p[1], q[1], false, false);
    return u32x4{a[0], a[1], b[0], b[1]};
}

template <int QT> struct RowRegs {
    u32x4 q0, q1;
    uint32_t h;
};

// Codes and header of this lane (see above) for the 128 columns of group g.  Blocks past the end of the row are read
// from the row's last one: their columns of x are zero.
template <int QT> __device__ inline void load_rows(gbytes row, int g, int c, int blocks, RowRegs<QT> &t) {
    using F = Fmt<QT>;
    int b = QT == QT_NF4 ? 2 * g + (c >> 1) : QT == QT_FP8_E4M3 ? g : 4 * g + c;
    b = b < blocks ? b : blocks - 1;
    const gbytes p = row + (int64_t)b * F::TS;
    const gbytes q = p + F::HDR + (QT == QT_NF4 ? 16 * (c & 1) : QT == QT_FP8_E4M3 ? 32 * c : 0);
    t.q0 = *(const __attribute__((address_space(1))) u32x4_a2 *)q;
    if constexpr (F::BITS == 8) t.q1 = *(const __attribute__((address_space(1))) u32x4_a2 *)(q + 16);
    if constexpr (F::HDR == 2) t.h = *(const __attribute__((address_space(1))) uint16_t *)p;
    else t.h = *(const __attribute__((address_space(1))) u32_a2 *)p;
}

// After this, step j has its codes where a tile of the tiled layout has those of sub-block j (4-bit: q0[j]; 8-bit: the
// two dwords 2j, 2j+1 of q0, q1) and its block's header in hb[j].
template <int QT> __device__ inline void arrange_rows(RowRegs<QT> &t, uint32_t (&hb)[4]) {
    if constexpr (QT == QT_FP8_E4M3) {
        hb[0] = hb[1] = hb[2] = hb[3] = t.h;
    } else {
        t.q0 = transpose_rows(t.q0);
        if constexpr (Fmt<QT>::BITS == 8) {
            const u32x4 a = t.q0, b = transpose_rows(t.q1);
            t.q0 = u32x4{a[0], b[0], a[1], b[1]};
            t.q1 = u32x4{a[2], b[2], a[3], b[3]};
        }
        spread_rows(t.h, hb);
    }
}

// Eight consecutive columns of x (chunk u of a row whose first column is a multiple of 128), stored into the row's
// LDS image in the order of the steps: lane c's operand of step j is the 16-byte unit j * 4 + c (of its 128 columns).
// `swizzle` (below 16) is xor-ed onto the unit: a kernel whose lanes read 16 rows 256 bytes apart passes the row, which
// spreads them over the LDS banks.
template <int QT> __device__ inline void store_x_rows(uint8_t *row, int u, const u32x4 &x, int swizzle = 0) {
    const int group = (u >> 4) * 16;
    auto unit = [&](int j, int c) __attribute__((always_inline)) { return row + (group + ((j * 4 + c) ^ swizzle)) * 16; };
    if constexpr (QT == QT_FP8_E4M3) {
        *(u32x4 *)unit(u & 3, (u >> 2) & 3) = x;
    } else if constexpr (QT == QT_SYM_INT8) {
        const int j = (u >> 2) & 3, c = 2 * (u & 1), half = ((u >> 1) & 1) * 8;
        *(u32x2 *)(unit(j, c) + half) = u32x2{x[0], x[1]};
        *(u32x2 *)(unit(j, c + 1) + half) = u32x2{x[2], x[3]};
    } else {
        const int j = QT == QT_NF4 ? ((u >> 3) & 1) * 2 + ((u >> 1) & 1) : (u >> 2) & 3, c = 2 * (u & 1);
        const int hi = (QT == QT_NF4 ? (u >> 2) & 1 : (u >> 1) & 1) * 4;
        uint8_t *const p = unit(j, c) + hi, *const q = unit(j, c + 1) + hi;
        *(uint32_t *)p = __builtin_amdgcn_perm(x[1], x[0], 0x05040100u);          // columns 0, 2
        *(uint32_t *)(p + 8) = __builtin_amdgcn_perm(x[1], x[0], 0x07060302u);    // columns 1, 3
        *(uint32_t *)q = __builtin_amdgcn_perm(x[3], x[2], 0x05040100u);          // columns 4, 6
        *(uint32_t *)(q + 8) = __builtin_amdgcn_perm(x[3], x[2], 0x07060302u);    // columns 5, 7
    }
}

}  // namespace lowbit
