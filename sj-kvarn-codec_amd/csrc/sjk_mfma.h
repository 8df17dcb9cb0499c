// sjk_mfma.h - matrix-core operand types and wavefront helpers shared by the attention kernels.
#pragma once
#include "sjk_dev.h"

namespace sjk {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef uint32_t u4 __attribute__((ext_vector_type(4)));
typedef uint32_t u2 __attribute__((ext_vector_type(2)));

SJK_DEV f4 mfma32(const u4 & a, const u4 & b, const f4 & c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, a), __builtin_bit_cast(h8, b), c, 0, 0, 0);
}

SJK_DEV f4 mfma16(const u2 & a, const u2 & b, const f4 & c) {
    return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(h4, a), __builtin_bit_cast(h4, b), c, 0, 0, 0);
}

SJK_DEV float h2f(uint32_t bits16) { return (float) __builtin_bit_cast(_Float16, (uint16_t) bits16); }

// (x0, x1) as fp16 pairs {hi, lo}: hi = RN16(x), lo = RN16(x - hi)
SJK_DEV u2 split2(float x0, float x1) {
    const _Float16 a = (_Float16) x0, b = (_Float16) x1;
    const _Float16 c = (_Float16) (x0 - (float) a), d = (_Float16) (x1 - (float) b);
    return u2{(uint32_t) __builtin_bit_cast(uint16_t, a) | ((uint32_t) __builtin_bit_cast(uint16_t, b) << 16),
              (uint32_t) __builtin_bit_cast(uint16_t, c) | ((uint32_t) __builtin_bit_cast(uint16_t, d) << 16)};
}

// sum / max over the four 16-lane rows of a wavefront (the MFMA lane groups g), (r0 + r1) + (r2 + r3), the
// same value in every lane
SJK_DEV float rows_sum(float v) {
    uint32_t a = __builtin_bit_cast(uint32_t, v), b = a;
    swap16(a, b);
    uint32_t c = __builtin_bit_cast(uint32_t, __builtin_bit_cast(float, a) + __builtin_bit_cast(float, b)), d = c;
    swap32(c, d);
    return __builtin_bit_cast(float, c) + __builtin_bit_cast(float, d);
}
SJK_DEV float rows_max(float v) {
    uint32_t a = __builtin_bit_cast(uint32_t, v), b = a;
    swap16(a, b);
    uint32_t c = __builtin_bit_cast(uint32_t, fmaxf(__builtin_bit_cast(float, a), __builtin_bit_cast(float, b))), d = c;
    swap32(c, d);
    return fmaxf(__builtin_bit_cast(float, c), __builtin_bit_cast(float, d));
}

// unsigned max over all 64 lanes: DPP rotations inside the rows, then across the rows
SJK_DEV uint32_t wave_umax(uint32_t v) {
    v = max(v, (uint32_t) __builtin_amdgcn_update_dpp(0, (int) v, 0x128, 0xF, 0xF, false));    // row_ror:8
    v = max(v, (uint32_t) __builtin_amdgcn_update_dpp(0, (int) v, 0x124, 0xF, 0xF, false));    // row_ror:4
    v = max(v, (uint32_t) __builtin_amdgcn_update_dpp(0, (int) v, 0x122, 0xF, 0xF, false));    // row_ror:2
    v = max(v, (uint32_t) __builtin_amdgcn_update_dpp(0, (int) v, 0x121, 0xF, 0xF, false));    // row_ror:1
    uint32_t a = v, b = v;
    swap16(a, b);
    uint32_t c = max(a, b), d = c;
    swap32(c, d);
    return max(c, d);
}

constexpr int A3_D = 256;

// record layout at head dimension D (256 unless given), G = 128 with BK / BV bits per K / V code
// (sj_kvarn.h:771-790): K payload | V payload | Kscale[D] | Kzero[D] | Ktok[G] | Vch[D] | Vscale[G] | Vzero[G]
template <int BK, int BV, int D = A3_D> struct RecLay {
    static constexpr int VPAY = 16 * D * BK, KSC = VPAY + 16 * D * BV, KZE = KSC + 2 * D, KTOK = KZE + 2 * D,
                         VCH = KTOK + 256, VSC = VCH + 2 * D, VZE = VSC + 256, BYTES = VZE + 256;
};

SJK_DEV float fma_lo(float a, uint32_t h2, float c) { return __builtin_fmaf(a, h2f(h2 & 0xFFFFu), c); }
SJK_DEV float fma_hi(float a, uint32_t h2, float c) { return __builtin_fmaf(a, h2f(h2 >> 16), c); }

// Power of two 2^k for the P' operands of one record: with vmax = max_t Vscale[t] in [2^(e-1), 2^e),
// P' = P * Vscale * 2^k (P <= 1, k = 14 - e) stays below 2^14 and the small weights stay clear of the
// fp16 subnormal range, where they would lose their low bits. Returns 2^k (uniform over
// the wave) and inv = 2^-k, by which the product is scaled back. vsc: the record's Vscale[128] in LDS.
SJK_DEV float pv_scale(const uint8_t * vsc, int lane, float & inv) {
    const uint32_t wv = *(const uint32_t *) (vsc + 4 * lane);       // Vscale of tokens 2 lane, 2 lane + 1 (>= 0)
    const uint32_t mx = wave_umax(max(wv & 0xFFFFu, wv >> 16));       // non-negative halves order like their bits
    const int e = __builtin_amdgcn_frexp_expf(h2f(mx));
    inv = __builtin_amdgcn_ldexpf(1.0f, e - 14);
    return __builtin_amdgcn_ldexpf(1.0f, 14 - e);
}

}  // namespace sjk
