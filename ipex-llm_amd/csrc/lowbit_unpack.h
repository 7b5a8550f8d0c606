// Codes as exact, unscaled MFMA operands: what the kernels that apply the block scale to the fp32 result share (the
// streaming kernel and the batch kernel for row-major weights).
#pragma once
#include "lowbit_mfma.h"

namespace lowbit {

// ---- codes of one sub-block (8 columns of this lane) -> B operand ----------
//
// The operand holds the *unscaled* code value (q - 8, q, int8, e4m3 value, nf4
// code-book entry); OFFSET says what constant is still folded in and has to
// be removed with the row sum of x (0 for every path below except bf16 4-bit).
// What the kernels use of this, and how, is Operand below.

template <int QT, typename AT> struct Unpack;

// 4-bit integer codes, fp16: 0x6400 | q is the half 1024 + q; 0x6400 | q << 4 is 1024 + 16 q.
template <> struct Unpack<QT_SYM_INT4, _Float16> {
    static constexpr float OFFSET = 0.0f;
    __device__ static f16x8 run(uint32_t v, const void *, uint32_t magic) {
        const f16x2 k1032 = {(_Float16)1032.0f, (_Float16)1032.0f};
        const f16x2 k16th = {(_Float16)0.0625f, (_Float16)0.0625f};
        const f16x2 k72 = {(_Float16)72.0f, (_Float16)72.0f};
        const uint32_t v8 = v >> 8;
        f16x2 t0 = __builtin_bit_cast(f16x2, and_or(v, 0x000f000fu, magic)) - k1032;
        f16x2 t1 = __builtin_elementwise_fma(__builtin_bit_cast(f16x2, and_or(v, 0x00f000f0u, magic)), k16th, -k72);
        f16x2 t2 = __builtin_bit_cast(f16x2, and_or(v8, 0x000f000fu, magic)) - k1032;
        f16x2 t3 = __builtin_elementwise_fma(__builtin_bit_cast(f16x2, and_or(v8, 0x00f000f0u, magic)), k16th, -k72);
        return f16x8{t0[0], t0[1], t1[0], t1[1], t2[0], t2[1], t3[0], t3[1]};
    }
};
template <> struct Unpack<QT_ASYM_INT4, _Float16> {
    static constexpr float OFFSET = 0.0f;
    __device__ static f16x8 run(uint32_t v, const void *, uint32_t magic) {
        const f16x2 k1024 = {(_Float16)1024.0f, (_Float16)1024.0f};
        const f16x2 k16th = {(_Float16)0.0625f, (_Float16)0.0625f};
        const f16x2 k64 = {(_Float16)64.0f, (_Float16)64.0f};
        const uint32_t v8 = v >> 8;
        f16x2 t0 = __builtin_bit_cast(f16x2, and_or(v, 0x000f000fu, magic)) - k1024;
        f16x2 t1 = __builtin_elementwise_fma(__builtin_bit_cast(f16x2, and_or(v, 0x00f000f0u, magic)), k16th, -k64);
        f16x2 t2 = __builtin_bit_cast(f16x2, and_or(v8, 0x000f000fu, magic)) - k1024;
        f16x2 t3 = __builtin_elementwise_fma(__builtin_bit_cast(f16x2, and_or(v8, 0x00f000f0u, magic)), k16th, -k64);
        return f16x8{t0[0], t0[1], t1[0], t1[1], t2[0], t2[1], t3[0], t3[1]};
    }
};
// 4-bit integer codes, bf16: 0x4300 | q is the bf16 128 + q (exact); the constant is removed
// afterwards through the row sum of x, which a second MFMA against all-ones provides.
template <int QT> struct UnpackInt4Bf16 {
    static constexpr float OFFSET = (QT == QT_SYM_INT4) ? 136.0f : 128.0f;
    __device__ static bf16x8 run(uint32_t v, const void *, uint32_t magic) {
        u32x4 t;
        t[0] = and_or(v, 0x000f000fu, magic);
        t[1] = and_or(v >> 4, 0x000f000fu, magic);
        t[2] = and_or(v >> 8, 0x000f000fu, magic);
        t[3] = and_or(v >> 12, 0x000f000fu, magic);
        return __builtin_bit_cast(bf16x8, t);
    }
};
template <> struct Unpack<QT_SYM_INT4, __bf16> : UnpackInt4Bf16<QT_SYM_INT4> {};
template <> struct Unpack<QT_ASYM_INT4, __bf16> : UnpackInt4Bf16<QT_ASYM_INT4> {};

// nf4: code-book lookup, two ways.
//   - From a 16-entry table in LDS: eight 2-byte reads and about twelve vector instructions per dword of codes.
//   - In registers: the 16 entries, already in the activation type, lie in two byte planes (low bytes, high bytes)
//     of four registers each; v_perm_b32 looks four codes up at a time in the eight bytes of a register pair -
//     entries 0..7 and 8..15 separately, a third v_perm_b32 picks per byte by the code's bit 3 - and two more
//     interleave the planes into 16-bit values: 21 vector instructions per dword of eight codes, no LDS access.
// Measured on one MI355X on the Llama-3-70B linear set (419 MB of nf4 weights, bf16): at M = 1 from LDS 115.9 us,
// in registers 123.0, half of the sub-blocks each way 117.7; at M = 16, where x takes its share of the LDS pipe,
// 171.4 / 156.7 / 165.6.  So up to four rows of x look up in LDS and more rows in registers.  Either way nf4 stays
// a quarter behind sym_int4 at the same bytes ([28672 x 8192] at M = 1: 31.7 against 25.5 us): the lookups are
// instructions the integer formats do not issue, whichever unit takes them.
struct Nf4Planes {
    uint32_t lo[4], hi[4];        // byte i % 4 of register i / 4 = low / high byte of entry i
    uint32_t k04, k0123;          // 0x04040404 and 0x03020100 in vector registers: as literals the two would need the
                                  // one constant slot of v_and_or_b32 twice
};
// PART 0 is the code book times SCALE rounded to AT, the next parts what the rounding of those before dropped.
template <typename AT, int PART, int SCALE> __device__ inline Nf4Planes nf4_planes() {
    Nf4Planes t = {};
#pragma unroll
    for (int i = 0; i < 16; i++) {                      // (constants: folded at compile time)
        const float v0 = NF4_CODEBOOK[i] * (float)SCALE, v1 = v0 - (float)to_at<AT>(v0), v2 = v1 - (float)to_at<AT>(v1);
        const uint32_t b = __builtin_bit_cast(uint16_t, to_at<AT>(PART == 0 ? v0 : PART == 1 ? v1 : v2));
        t.lo[i / 4] |= (b & 0xffu) << (8 * (i % 4));
        t.hi[i / 4] |= (b >> 8) << (8 * (i % 4));
    }
    asm("v_mov_b32 %0, 0x04040404" : "=v"(t.k04));
    asm("v_mov_b32 %0, 0x03020100" : "=v"(t.k0123));
    return t;
}
template <typename AT> struct Unpack<QT_NF4, AT> {
    static constexpr float OFFSET = 0.0f;
    // four codes, one per byte of `sel` (bits 0..2) and `mrg` (0x03020100 + 4 * bit 3 per byte) -> one byte plane
    __device__ static uint32_t plane4(const uint32_t (&p)[4], uint32_t sel, uint32_t mrg) {
        return __builtin_amdgcn_perm(__builtin_amdgcn_perm(p[3], p[2], sel), __builtin_amdgcn_perm(p[1], p[0], sel), mrg);
    }
    __device__ static typename Vec8<AT>::type run(uint32_t v, const void *planes_, uint32_t) {
        const Nf4Planes &t = *(const Nf4Planes *)planes_;
        // nibbles 0, 2, 4, 6 (columns 0, 4, 1, 5) are the low nibbles of the four bytes, 1, 3, 5, 7 (columns 2, 6,
        // 3, 7) the high ones
        const uint32_t sel_e = v & 0x07070707u, mrg_e = and_or(v >> 1, t.k04, t.k0123);
        const uint32_t sel_o = (v >> 4) & 0x07070707u, mrg_o = and_or(v >> 5, t.k04, t.k0123);
        const uint32_t lo_e = plane4(t.lo, sel_e, mrg_e), hi_e = plane4(t.hi, sel_e, mrg_e);
        const uint32_t lo_o = plane4(t.lo, sel_o, mrg_o), hi_o = plane4(t.hi, sel_o, mrg_o);
        u32x4 r;
        r[0] = __builtin_amdgcn_perm(hi_e, lo_e, 0x06020400u);      // columns 0, 1: bytes 0 and 2 of the even set
        r[1] = __builtin_amdgcn_perm(hi_o, lo_o, 0x06020400u);      // columns 2, 3
        r[2] = __builtin_amdgcn_perm(hi_e, lo_e, 0x07030501u);      // columns 4, 5: bytes 1 and 3
        r[3] = __builtin_amdgcn_perm(hi_o, lo_o, 0x07030501u);      // columns 6, 7
        return __builtin_bit_cast(typename Vec8<AT>::type, r);
    }
    __device__ static typename Vec8<AT>::type run_lds(uint32_t v, const AT *lut) {
        typename Vec8<AT>::type r;
        r[0] = lut[v & 0xf]; r[2] = lut[(v >> 4) & 0xf]; r[4] = lut[(v >> 8) & 0xf]; r[6] = lut[(v >> 12) & 0xf];
        r[1] = lut[(v >> 16) & 0xf]; r[3] = lut[(v >> 20) & 0xf]; r[5] = lut[(v >> 24) & 0xf]; r[7] = lut[v >> 28];
        return r;
    }
};

// 4-bit integer codes centred, in bf16: (q - 8) / 16, which v_cvt_off_f32_i4 makes of the low four bits of a byte whose
// bit 3 is flipped.  14 instructions per dword of codes (the or-ed pattern of UnpackInt4Bf16: 7; a lookup as nf4's: 21).
__device__ inline bf16x8 centred_bf16(uint32_t v) {
    const uint32_t lo = v ^ 0x88888888u;
    uint32_t hi = lo >> 4;
    asm("" : "+v"(hi));                                 // (its bytes are then picked by the conversion itself)
    auto code = [](uint32_t byte) { return (__bf16)__builtin_amdgcn_cvt_off_f32_i4((int)byte); };
    return bf16x8{code(lo), code((lo >> 16) & 0xff), code(hi), code((hi >> 16) & 0xff),
                  code((lo >> 8) & 0xff), code(lo >> 24), code((hi >> 8) & 0xff), code(hi >> 24)};
}

// 8-bit codes: two dwords (columns 0..3, 4..7).
template <int QT, typename AT> struct Unpack8;
template <> struct Unpack8<QT_SYM_INT8, _Float16> {
    __device__ static f16x8 run(uint32_t lo, uint32_t hi) {
        // byte ^ 0x80 = q + 128 (unsigned); 0x6400 | u is the half 1024 + u
        const f16x2 k1152 = {(_Float16)1152.0f, (_Float16)1152.0f};
        const uint32_t a = lo ^ 0x80808080u, b = hi ^ 0x80808080u;
        const uint32_t c64 = 0x64646464u;
        f16x2 t0 = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(c64, a, 0x04010400u)) - k1152;
        f16x2 t1 = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(c64, a, 0x04030402u)) - k1152;
        f16x2 t2 = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(c64, b, 0x04010400u)) - k1152;
        f16x2 t3 = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(c64, b, 0x04030402u)) - k1152;
        return f16x8{t0[0], t0[1], t1[0], t1[1], t2[0], t2[1], t3[0], t3[1]};
    }
};
template <> struct Unpack8<QT_SYM_INT8, __bf16> {
    __device__ static bf16x8 run(uint32_t lo, uint32_t hi) {
        bf16x8 r;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            r[i] = (__bf16)(float)(int8_t)(lo >> (8 * i));      // |q| <= 128: exact in bf16
            r[4 + i] = (__bf16)(float)(int8_t)(hi >> (8 * i));
        }
        return r;
    }
};
template <> struct Unpack8<QT_FP8_E4M3, _Float16> {
    __device__ static f16x8 run(uint32_t lo, uint32_t hi) {
        f16x2 t0 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(lo, 1.0f, false);
        f16x2 t1 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(lo, 1.0f, true);
        f16x2 t2 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(hi, 1.0f, false);
        f16x2 t3 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(hi, 1.0f, true);
        return f16x8{t0[0], t0[1], t1[0], t1[1], t2[0], t2[1], t3[0], t3[1]};
    }
};
template <> struct Unpack8<QT_FP8_E4M3, __bf16> {
    __device__ static bf16x8 run(uint32_t lo, uint32_t hi) {
        bf16x2 t0 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.0f, false);
        bf16x2 t1 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.0f, true);
        bf16x2 t2 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.0f, false);
        bf16x2 t3 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.0f, true);
        return bf16x8{t0[0], t0[1], t1[0], t1[1], t2[0], t2[1], t3[0], t3[1]};
    }
};

// The MFMA operand that codes become in a kernel, and what the kernel has to know about it.
//   PARTS   16-bit operands whose sum is the code's value, one MFMA each
//   OFFSET  constant still in the value, removed through the row sum of x (NEED_S)
// Tiled weights with 16-bit activations: one part, the constant as Unpack has it.  F32 (float32 activations) and ROWS
// (row-major weights, which were decoded to fp32 before the product): operands that keep the result's precision.
//   4-bit integers are centred, q - 8.  With the 128 or 136 that Unpack leaves in bf16, fp32 sums some 17 times larger
//     cancel, and x's second plane loses bits beside the first one's: float32 activations were off by 3.8e-6 of the
//     result's norm in place of 2.5e-6, and ten times as many bf16 results were not the nearest one.  asym_int4's minimum, mostly near -7.5 scales, goes with the 8, and a step's two
//     terms meet before they go to the sum, which is then rounded once a step (fp16 results of 8640 columns that are not
//     the nearest: 1.23 in a thousand with two FMAs, 0.98 this way, 1.05 from weights in fp32).
//   nf4's code book has 24 mantissa bits.  ROWS: three parts in bf16, which hold it exactly (two are off by up to 5e-6 of an
//     entry: 3.5e-6 of the result's norm with float32 activations, 2.6 bf16 results in a thousand not the nearest one, 0.17
//     from weights in fp32), two in fp16 with the book scaled by 2^14, which keeps the second one clear of fp16's subnormal
//     numbers: three of the 16 entries are then off by one in the 24th bit, the others exact.  Tiled with F32: two parts.
template <int QT, typename AT, bool F32, bool ROWS> struct Operand {
    using V8 = typename Vec8<AT>::type;
    static constexpr bool NF4 = QT == QT_NF4, INT4 = QT == QT_SYM_INT4 || QT == QT_ASYM_INT4;
    static constexpr bool CENTRED = INT4 && (ROWS || F32), CENTRED_BF16 = CENTRED && __is_same(AT, __bf16);
    static constexpr int PARTS = !NF4 ? 1 : ROWS ? (__is_same(AT, __bf16) ? 3 : 2) : F32 ? 2 : 1;
    static constexpr int NF4_SCALE = NF4 && ROWS && __is_same(AT, _Float16) ? 1 << 14 : 1;
    static constexpr float offset() {
        if constexpr (CENTRED) return QT == QT_ASYM_INT4 ? -8.0f : 0.0f;
        else if constexpr (INT4) return Unpack<QT, AT>::OFFSET;
        else return 0.0f;
    }
    static constexpr float OFFSET = offset();
    static constexpr bool NEED_S = QT == QT_ASYM_INT4 || OFFSET != 0.0f;

    Nf4Planes planes[PARTS];
    // exponent pattern OR-ed onto 4-bit codes (fp16 1024, bf16 128), held in a vector register: as a literal it would share
    // the instruction's one constant slot with the nibble mask and split every v_and_or_b32 into an AND and an OR
    uint32_t magic;

    __device__ Operand() {
        if constexpr (NF4) planes[0] = nf4_planes<AT, 0, NF4_SCALE>();
        if constexpr (PARTS > 1) planes[1] = nf4_planes<AT, 1, NF4_SCALE>();
        if constexpr (PARTS > 2) planes[2] = nf4_planes<AT, 2, NF4_SCALE>();
        if constexpr (__is_same(AT, _Float16)) asm("v_mov_b32 %0, 0x64006400" : "=v"(magic));
        else asm("v_mov_b32 %0, 0x43004300" : "=v"(magic));
    }
    // what a step's product is to be multiplied by, from its block's scale
    __device__ static float scale(float d) { return CENTRED_BF16 ? 16.0f * d : d * (1.0f / NF4_SCALE); }
    // sum + d * p + e * s: that times the step's product, e (see OFFSET) times the row sum of x
    __device__ static float add(float sum, float d, float p, float e, float s) {
        if constexpr (!NEED_S) return fmaf(d, p, sum);
        else if constexpr (CENTRED) return sum + fmaf(e, s, d * p);
        else return fmaf(e, s, fmaf(d, p, sum));
    }
    // a step's product; al: what x's first plane leaves (F32).  The largest first: an MFMA drops more of a small sum that it
    // is given beside large products than of small products beside a large sum (fp16, 8640 columns: 1.48 in a thousand not
    // the nearest result the other way round, 1.14 this way).  The smallest parts of both are below fp32.
    __device__ static f32x4 product(const V8 &a, const V8 &al, const V8 (&b)[PARTS], f32x4 p = {0.0f, 0.0f, 0.0f, 0.0f}) {
#pragma unroll
        for (int part = 0; part < PARTS; part++) {
            p = mfma16(a, b[part], p);
            if (F32 && part < 2) p = mfma16(al, b[part], p);
        }
        return p;
    }
    // part p of step j's eight codes; t: TileRegs, or RowRegs after arrange_rows
    template <typename Regs> __device__ V8 get(const Regs &t, int j, int p) const {
        if constexpr (NF4) return Unpack<QT_NF4, AT>::run(t.q0[j], &planes[p], magic);
        else if constexpr (CENTRED_BF16) return centred_bf16(t.q0[j]);
        else if constexpr (CENTRED) return Unpack<QT_SYM_INT4, AT>::run(t.q0[j], nullptr, magic);
        else if constexpr (INT4) return Unpack<QT, AT>::run(t.q0[j], nullptr, magic);
        else if (j < 2) return Unpack8<QT, AT>::run(t.q0[(2 * j) & 3], t.q0[(2 * j + 1) & 3]);
        else return Unpack8<QT, AT>::run(t.q1[(2 * j) & 3], t.q1[(2 * j + 1) & 3]);
    }
};

template <typename AT> __device__ inline typename Vec8<AT>::type ones8() {
    typename Vec8<AT>::type r;
#pragma unroll
    for (int i = 0; i < 8; i++) r[i] = to_at<AT>(1.0f);
    return r;
}

// Eight floats -> their bf16 values and those of what the rounding dropped.  inf / nan stay in the first plane only, or, without KEEP,
// make NaN of the second: three of six instructions less, for kernels that compute a result that is not finite once more (below).
template <bool KEEP = true> __device__ inline void split_f32(const u32x4 &a, const u32x4 &b, u32x4 &hi, u32x4 &lo) {
    bf16x8 h, l;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const float v = __builtin_bit_cast(float, i < 4 ? a[i] : b[i - 4]);
        h[i] = (__bf16)v;                                   // round to nearest even
        const float r = v - (float)h[i];                    // exact: both share the leading bits
        l[i] = !KEEP || (r - r) == 0.0f ? (__bf16)r : (__bf16)0.0f;
    }
    hi = __builtin_bit_cast(u32x4, h);
    lo = __builtin_bit_cast(u32x4, l);
}

// ---- results that are not finite
//
// The kernels multiply activations by codes and apply scale, minimum and the parts of a value afterwards.  An infinity among
// the activations then meets a code of zero whose weight is not zero, terms d * inf and e * inf of opposite signs, or parts
// of opposite signs: NaN, where the weight times it is a signed infinity.  (And sums of codes can overflow where the weights'
// do not.)  So a kernel computes a result that is not finite once more: from the columns of x that are not finite and their
// weights, decoded to fp32, or, where x is finite, from all of them.  A test per result; time goes only into calls that have
// one (333 rows on [3200 x 8640] in sym_int4, an infinity in every row: 1.7 ms, in none: 0.05).

// the weight in row n, column k
template <int QT, bool ROWS> __device__ inline float weight_fp32(const uint8_t *w, int64_t n, int64_t K, int64_t k) {
    using F = Fmt<QT>;
    const uint8_t *codes, *hdr;
    int nibble = 0;
    if constexpr (ROWS) {                                    // block k / QK of the row
        hdr = w + (n * (K / F::QK) + k / F::QK) * F::TS;
        const int i = (int)(k % F::QK);
        codes = hdr + F::HDR + (F::BITS == 8 ? i : i % (F::QK / 2));
        nibble = i / (F::QK / 2);
    } else {                                                 // sub-block j of its tile, column group c, see lowbit_formats.h
        const int r = (int)(n % TILE_ROWS), j = (int)(k / 32 % 4), c = (int)(k % 32 / 8), i = (int)(k % 8);
        const uint8_t *tile = w + tile_offset<QT>(n, K, (int)(k / 32));
        hdr = tile + tile_hdr_offset<QT>(r, j);
        codes = tile + (c * 16 + r) * 16 + (F::BITS == 8 ? j / 2 * 1024 + j % 2 * 8 + i : j * 4 + ((i & 1) * 4 + i / 2) / 2);
        nibble = i / 2 % 2;
    }
    uint32_t h = *(const uint16_t *)hdr;
    if constexpr (F::HDR == 4) h |= (uint32_t)((const uint16_t *)hdr)[1] << 16;
    float d, m;
    hdr_to_scale<QT>(h, d, m);
    return decode<QT>(F::BITS == 8 ? *codes : (*codes >> nibble * 4) & 15u, d, m);
}

// x: the row, 16-byte aligned; K a multiple of 8
template <int QT, bool ROWS, typename ET>
__device__ inline float dot_fp32(const ET *x, const uint8_t *w, int64_t n, int64_t K) {
    typedef ET V8 __attribute__((ext_vector_type(8), aligned(16)));
    float sum = 0.0f;
    bool all_finite = true;
    for (int64_t k = 0; k < K && sum == sum; k += 8) {
        const V8 v = *(const V8 *)(x + k);
        uint32_t odd = 0;
#pragma unroll
        for (int i = 0; i < 8; i++) odd |= __builtin_isfinite((float)v[i]) ? 0u : 1u << i;
        for (; odd; odd &= odd - 1) {
            const int64_t at = k + __builtin_ctz(odd);
            sum = fmaf((float)x[at], weight_fp32<QT, ROWS>(w, n, K, at), sum);
            all_finite = false;
        }
    }
    if (all_finite)
        for (int64_t k = 0; k < K && sum == sum; k++) sum = fmaf((float)x[k], weight_fp32<QT, ROWS>(w, n, K, k), sum);
    return sum;
}

// activation of the gate branch: 0 = SiLU, 1 = GELU in its tanh form (what Gemma uses)
__device__ inline float gate_act(float g, int act) {
    if (act == 0) return g / (1.0f + __expf(-g));
    const float t = tanhf(0.7978845608028654f * (g + 0.044715f * g * g * g));
    return 0.5f * g * (1.0f + t);
}

}  // namespace lowbit
