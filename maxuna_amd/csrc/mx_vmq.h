// Weight operands of v_mfma_f32_16x16x32_f16 from whole super-blocks in LDS,
// shared by the verify tiles (mx_vmm.hip) and the stationary-activation expert
// matmul (mx_gst.hip): lane l holds row l % 16 of a 16-row block and K quarter
// q = l / 16.
#pragma once

#include "mx_wb.h"

namespace mx {
namespace {

// Q6_K half super-block PAR of the lane's row from its slot (the block's span from
// the 16-byte-aligned address below it; ph = the block's phase): 8 bytes of each
// field, the lane's values 32 P + 8 q + [0, 8) of step P (part P of the half).  The
// same weights as WB<kQ6_K>, whose lanes hold 16 bytes of a field for the 32 x 32
// layout: here half of them would be read, shifted and selected away (the Q6_K
// verify tiles 116 -> 108 us in a 16-token block of hidden 4096, ff 1536; mx_gst.hip at 512
// tokens 478 -> 437).
struct VmQ6 {
    uint2 lo, hi, qh;   // ql[64 PAR + 8 q, +8), ql[64 PAR + 32 + 8 q, +8), qh[32 PAR + 8 q, +8)
    uint2 sc;           // scales[8 PAR, +8)
    uint32_t d;
    float d1[4], c1[4]; // d * sc and -1056 * d * sc of the lane's 16-value group of each part
    template <int PAR> __device__ __forceinline__ void load(const uint8_t *slot, int q, uint32_t ph) {
        lo = lds8_a2(slot, ph + 64 * PAR + 8 * q);
        hi = lds8_a2(slot, ph + 64 * PAR + 32 + 8 * q);
        qh = lds8_a2(slot, ph + 128 + 32 * PAR + 8 * q);
        sc = lds8_a2(slot, ph + 192 + 8 * PAR);
        d = *reinterpret_cast<const uint16_t *>(slot + ph + 208);
    }
    __device__ __forceinline__ void prep(int kh) {
        const float df = h2f((uint16_t)d);
#pragma unroll
        for (int p = 0; p < 4; p++) {  // scale 8 PAR + 2 p + kh
            const uint32_t word = p < 2 ? sc.x : sc.y;
            d1[p] = df * (float)(int)__builtin_amdgcn_sbfe((int)word, 16 * (p & 1) + 8 * kh, 8);
            c1[p] = -1056.0f * d1[p];
        }
    }
    template <int P> __device__ __forceinline__ half8_t step() const {
        constexpr int S = 4 * (P >> 1);
        const uint2 v = (P & 1) ? hi : lo;
        auto top = [](uint32_t w) {
            return P < 2 ? (w << (4 - 2 * P)) & 0x30303030u : P == 2 ? w & 0x30303030u : (w >> 2) & 0x30303030u;
        };
        return dq8_q6(((v.x >> S) & 0x0F0F0F0Fu) | top(qh.x), ((v.y >> S) & 0x0F0F0F0Fu) | top(qh.y), d1[P], c1[P]);
    }
};

// Q4_K half super-block `PAR` of the lane's row for the sub-block-per-lane
// order: sub-block j = 4 PAR + q (32 values, one 6-bit scale and min).  Word i of
// its 32 quant bytes holds values 4 i .. 4 i + 3 in the lane's nibble (low for
// even q, high for odd q).  One and-or against the f16 exponent 0x6400 turns a
// word into the f16 pair 1024 + q of values 4 i and 4 i + 2 (the word shifted by
// a byte: 4 i + 1 and 4 i + 3), so step P gives values 8 P + {0, 2, 1, 3, 4, 6,
// 5, 7}: the A rows are stored in that order (launch_to_f16_rows with perm).  A
// high nibble reads as 1024 + 16 q, so odd sub-blocks take d1 / 16 (exact); each
// value is the f32 fma (1024 + q) d1 + c rounded to f16 once, as in WB<kQ4_K>.
struct VmQ4 {
    uint32_t w[8];  // the quant bytes of values 4 i .. 4 i + 3 in word i
    uint32_t m;     // the lane's nibble of bytes 0 and 2: 0x000F000F or 0x00F000F0
    float d1, c1;   // d * sc (/ 16 for a high nibble) and -dmin * m - 1024 * d1
    template <int PAR> __device__ __forceinline__ void load(const uint8_t *slot, int q) {
        const uint4 h = ld_w4(slot);  // d, dmin | scales[12]
        const uint8_t *qs = slot + 16 + 64 * PAR + 32 * (q >> 1); // the sub-block pair's 32 bytes
        const uint4 a = ld_w4(qs);
        const uint4 b = ld_w4(qs + 16);
        w[0] = a.x; w[1] = a.y; w[2] = a.z; w[3] = a.w;
        w[4] = b.x; w[5] = b.y; w[6] = b.z; w[7] = b.w;
        m = (q & 1) ? 0x00F000F0u : 0x000F000Fu;
        // get_scale_min_k4 of sub-block j (q4k_scale_min) with j = 4 PAR + q
        const uint32_t o = 8u * (uint32_t)q;
        uint32_t sc, mn;
        if constexpr (PAR == 0) {
            sc = __builtin_amdgcn_ubfe(h.y, o, 6);
            mn = __builtin_amdgcn_ubfe(h.z, o, 6);
        } else {
            const uint32_t b8 = __builtin_amdgcn_ubfe(h.w, o, 8);
            sc = (b8 & 0xFu) | (__builtin_amdgcn_ubfe(h.y, o + 6, 2) << 4);
            mn = (b8 >> 4) | (__builtin_amdgcn_ubfe(h.z, o + 6, 2) << 4);
        }
        const float d = h2f((uint16_t)(h.x & 0xFFFFu)), dmin = h2f((uint16_t)(h.x >> 16));
        d1 = d * (float)sc * ((q & 1) ? 0.0625f : 1.0f);
        c1 = __builtin_fmaf(-1024.0f, d1, -(dmin * (float)mn));
    }
    __device__ __forceinline__ half8_t step(int P) const {
        const uint32_t r0 = w[2 * P], r1 = w[2 * P + 1];
        const half2_t x[4] = {__builtin_bit_cast(half2_t, (r0 & m) | 0x64006400u),
                              __builtin_bit_cast(half2_t, ((r0 >> 8) & m) | 0x64006400u),
                              __builtin_bit_cast(half2_t, (r1 & m) | 0x64006400u),
                              __builtin_bit_cast(half2_t, ((r1 >> 8) & m) | 0x64006400u)};
        half2_t y[4];
#pragma unroll
        for (int i = 0; i < 4; i++) y[i] = mix2(x[i], d1, c1);
        return pk_join(y);
    }
};

}  // namespace
}  // namespace mx
