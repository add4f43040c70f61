// Plain quantised mat-vec for several tokens at once (the vocabulary projection of a
// verified block or of a small batch; replaces ops::mv_id::mul_mv, mv_id.rs:54-56, for
// those), and for one token of rows that the ring kernel does not take
// (mv_tokens_takes).
//
// The per-token mat-vecs read and unpack the matrix once per token.  Here the
// activations stay put and the weights stream past them once: every wave of a
// workgroup owns one super-block (256 values) of K and holds 16 tokens'
// activations for it in registers as MFMA operands; the workgroup walks 16-row
// tiles of the matrix, each wave contracting its K share of the tile
// (v_mfma_f32_16x16x32_f16), and the waves' partial sums meet in LDS in wave
// order.  Rows of more than MT_WAVES super-blocks run as several launches, each
// adding its K range to dst (several super-blocks in a wave's registers spill).
//
// Precision (f32 class).  The weights enter as their integer quants, exact in
// f16, and the scales are applied to each scale group's sum in f32.  Every
// activation is two f16 pieces, hi + lo, of the value times a power of two (per
// token and super-block, the largest magnitude in [2^14, 2^15)): hi carries 11
// bits and lo the next 11, so a value is held to 2^-23 of itself, or 2^-40 of the
// super-block's largest.  Products are exact in f32 and the sums are f32.
//   Q4_K, Q5_K, Q8_0 (32-value scale groups): a step is 32 K values, contracted
//     with lo, then with hi on top of it.
//   Q6_K (16-value scale groups): a step's 32 values are two groups; K is filled
//     with hi and lo side by side (lane quarters 0, 1 and 2, 3), and the weights of
//     either group are copied to both lane halves (v_permlane32_swap), so one MFMA
//     gives one group's sum.
//
// Weight bytes: a wave copies the 16-byte chunks that cover its super-block of
// each of the tile's 16 rows into its own LDS (two buffers), reads the lanes'
// words into registers, and issues the copy of the tile after the next into the
// same buffer before it computes.
//
// Bound by instruction issue (68% of the SIMD cycles): about 40 VALU per step of 512
// weights (unpacking, the copies to both lane halves, the scales).  lm_head [100352 x 3072] Q6_K at 16
// tokens: 503 us as 16 mat-vecs, 82 us here (3.1 TB/s of weights); relative error
// against 64 bits 2.4e-7 before, 1.2e-7 here.  One stage buffer per wave took 91 us.
#include "mx_launch.h"
#include "mx_dma.h"
#include "mx_wb.h"

namespace mx {
namespace {

constexpr int MT_WAVES = 12;  // waves of a workgroup at most: 3 per SIMD, 168 registers
constexpr int MT_TOK = 16;  // tokens per pass over the matrix
constexpr int MT_ROWS = 16; // rows per tile

// 16-byte chunks copied per row and super-block; the LDS slot of a row is as long
// (16 rows on distinct banks); 2-byte-aligned types: the aligned span
template <int DT> struct MtBlk;
template <> struct MtBlk<kQ4_K> { static constexpr int BLK = 144, CPR = 9; };
template <> struct MtBlk<kQ5_K> { static constexpr int BLK = 176, CPR = 11; };
template <> struct MtBlk<kQ6_K> { static constexpr int BLK = 210, CPR = 15; };
template <> struct MtBlk<kQ8_0> { static constexpr int BLK = 272, CPR = 19; };

// f16 (1024 + byte) of bytes 0..3 of a and b, minus off (both exact)
__device__ __forceinline__ half8_t bytes_f16(uint32_t a, uint32_t b, float off) {
    const half2_t o = {(_Float16)off, (_Float16)off};
    auto two = [&](uint32_t w, uint32_t sel) {
        return __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, w, sel)) - o;
    };
    const half2_t x0 = two(a, 0x04010400u), x1 = two(a, 0x04030402u), x2 = two(b, 0x04010400u), x3 = two(b, 0x04030402u);
    return half8_t{x0[0], x0[1], x1[0], x1[1], x2[0], x2[1], x3[0], x3[1]};
}

// One super-block of the lane's row n = lane % 16: quants of K quarter q = lane /
// 16 (values 8 q .. 8 q + 7 of each step of 32), and the row's scales.
// b(J): the step's quants as f16.  Step J covers values 32 J .. 32 J + 31.
template <int DT> struct MtW;
// a K-quant sub-block's weight s q - dmin m as s (q - mid) + c: the quants enter
// centred, so the two terms do not cancel for centred weights
template <int J> __device__ __forceinline__ void kmin_scales(const uint4 &h, float mid, float &s, float &c) {
    uint32_t sc, mn;
    q4k_scale_min(J, h.y, h.z, h.w, sc, mn);
    s = h2f((uint16_t)(h.x & 0xFFFFu)) * (float)sc;
    c = __builtin_fmaf(mid, s, -(h2f((uint16_t)(h.x >> 16)) * (float)mn));
}
template <> struct MtW<kQ4_K> {
    static constexpr int kMid = 8;
    uint4 h;
    uint32_t w[8];  // pair i: words 2 i, 2 i + 1
    __device__ __forceinline__ void load(const uint8_t *slot, uint32_t, int q) {
        h = *reinterpret_cast<const uint4 *>(slot);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint2 v = *reinterpret_cast<const uint2 *>(slot + 16 + 32 * i + 8 * q);
            w[2 * i] = v.x;
            w[2 * i + 1] = v.y;
        }
    }
    template <int J> __device__ __forceinline__ half8_t b() const {
        constexpr uint32_t S = 4 * (J & 1);
        const uint32_t a0 = (w[2 * (J >> 1)] >> S) & 0x0F0F0F0Fu, a1 = (w[2 * (J >> 1) + 1] >> S) & 0x0F0F0F0Fu;
        return bytes_f16(a0, a1, 1024.f + kMid);
    }
    template <int J> __device__ __forceinline__ void scales(float &s, float &c) const {
        kmin_scales<J>(h, (float)kMid, s, c);
    }
};
template <> struct MtW<kQ5_K> {
    static constexpr int kMid = 16;
    uint4 h;
    uint32_t w[8], hb[2];
    __device__ __forceinline__ void load(const uint8_t *slot, uint32_t, int q) {
        h = *reinterpret_cast<const uint4 *>(slot);
        const uint2 b5 = *reinterpret_cast<const uint2 *>(slot + 16 + 8 * q);
        hb[0] = b5.x;
        hb[1] = b5.y;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint2 v = *reinterpret_cast<const uint2 *>(slot + 48 + 32 * i + 8 * q);
            w[2 * i] = v.x;
            w[2 * i + 1] = v.y;
        }
    }
    template <int J> __device__ __forceinline__ half8_t b() const {
        constexpr uint32_t S = 4 * (J & 1);
        const uint32_t a0 = ((w[2 * (J >> 1)] >> S) & 0x0F0F0F0Fu) | (((hb[0] >> J) & 0x01010101u) << 4);
        const uint32_t a1 = ((w[2 * (J >> 1) + 1] >> S) & 0x0F0F0F0Fu) | (((hb[1] >> J) & 0x01010101u) << 4);
        return bytes_f16(a0, a1, 1024.f + kMid);
    }
    template <int J> __device__ __forceinline__ void scales(float &s, float &c) const {
        kmin_scales<J>(h, (float)kMid, s, c);
    }
};
template <> struct MtW<kQ6_K> {
    uint2 lo[2], hi[2], qh[2];  // per half: ql[64 n + 8 q, +8), ql[64 n + 32 + 8 q, +8), qh[32 n + 8 q, +8)
    uint2 sc[2];                // scales[8 n, +8)
    uint32_t d;
    __device__ __forceinline__ void load(const uint8_t *slot, uint32_t ph, int q) {
#pragma unroll
        for (int n = 0; n < 2; n++) {
            lo[n] = lds8_a2(slot, ph + 64 * n + 8 * q);
            hi[n] = lds8_a2(slot, ph + 64 * n + 32 + 8 * q);
            qh[n] = lds8_a2(slot, ph + 128 + 32 * n + 8 * q);
            sc[n] = lds8_a2(slot, ph + 192 + 8 * n);
        }
        d = *reinterpret_cast<const uint16_t *>(slot + ph + 208);
    }
    // step J = part p of half n (positions 128 n + 32 p): low nibbles of lo, hi for
    // p = 0, 1, high nibbles for p = 2, 3, and bits 2 p of qh
    template <int J> __device__ __forceinline__ half8_t b() const {
        constexpr int n = J >> 2, p = J & 3, S = 4 * (p >> 1);
        const uint2 v = (p & 1) ? hi[n] : lo[n];
        auto top = [&](uint32_t w) {
            return p < 2 ? (w << (4 - 2 * p)) & 0x30303030u : p == 2 ? w & 0x30303030u : (w >> 2) & 0x30303030u;
        };
        return bytes_f16(((v.x >> S) & 0x0F0F0F0Fu) | top(qh[n].x), ((v.y >> S) & 0x0F0F0F0Fu) | top(qh[n].y), 1056.f);
    }
    // the int8 scale of group g (16 values) of step J
    template <int J, int G> __device__ __forceinline__ float scale() const {
        constexpr int n = J >> 2, p = J & 3, j = 2 * p + G;
        return (float)(int)__builtin_amdgcn_sbfe((int)(j < 4 ? sc[n].x : sc[n].y), 8 * (j & 3), 8);
    }
};
template <> struct MtW<kQ8_0> {
    uint2 v[8];
    uint32_t d[8];
    __device__ __forceinline__ void load(const uint8_t *slot, uint32_t ph, int q) {
#pragma unroll
        for (int j = 0; j < 8; j++) {
            v[j] = lds8_a2(slot, ph + 34 * j + 2 + 8 * q);
            d[j] = *reinterpret_cast<const uint16_t *>(slot + ph + 34 * j);
        }
    }
    template <int J> __device__ __forceinline__ half8_t b() const {
        return bytes_f16(v[J].x ^ 0x80808080u, v[J].y ^ 0x80808080u, 1152.f);
    }
    template <int J> __device__ __forceinline__ void scales(float &s, float &c) const {
        s = h2f((uint16_t)d[J]);
        c = 0.f;
    }
};

template <int DT> constexpr bool kMin = DT == kQ4_K || DT == kQ5_K;

}  // namespace

struct MtArgs {
    const uint8_t *w;
    int64_t row_bytes;
    int n_out, k, t;
    const float *x;  // [t, k]
    float *dst;      // [t, n_out]
    int sb;          // first super-block of this launch's K range (one per wave)
};

// LDS: two stage buffers (16 rows' chunks) per wave, and the fixed arrays
template <int DT> struct MtLds {
    static constexpr int STAGE = MT_ROWS * MtBlk<DT>::CPR * 16;
    static constexpr int FIXED = MT_WAVES * (2 * 256 + MT_TOK + (kMin<DT> ? 8 * MT_TOK : 0)) * 4;
    static constexpr int bytes(int waves) { return waves * 2 * STAGE; }
};

// ADD: dst holds the sums of the K ranges before this one
template <int DT, bool ADD>
__global__ void __launch_bounds__(64 * MT_WAVES) k_mv_tokens(MtArgs a) {
    using B = MtBlk<DT>;
    constexpr int CPR = B::CPR, SLOT = 16 * CPR, POS = MT_ROWS * CPR, NI = (POS + 63) / 64;
    // the stage buffers (two per wave) apart from what is read while copies into them
    // are in flight, so that the compiler sees that the copies do not feed those reads
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    __shared__ __attribute__((aligned(16))) float sRed[2][MT_WAVES][256];  // partial sums, two parities
    __shared__ __attribute__((aligned(16))) float sTs[MT_WAVES][MT_TOK];    // token scales
    __shared__ __attribute__((aligned(16))) float sSum[kMin<DT> ? MT_WAVES : 1][8][MT_TOK];  // sums of 32 values
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), W = blockDim.x >> 6;
    const int n = lane & 15, q = lane >> 4;
    const int sb = a.sb + wave;  // this wave's super-block
    const int tok0 = blockIdx.y * MT_TOK;
    const int tiles = (a.n_out + MT_ROWS - 1) / MT_ROWS, G = (int)gridDim.x;
    constexpr int STAGE = MtLds<DT>::STAGE;
    uint8_t *const buf0 = lds + wave * (2 * STAGE), *const buf1 = buf0 + STAGE;

    // the copy of the wave's super-block of a tile's rows: the aligned chunks that
    // cover each row's block, the last one repeated.  16 rows are a multiple of 16
    // bytes, so every tile starts at the same phase and a lane's chunk keeps its
    // offset from the tile's first aligned byte; in a last partial tile the chunks
    // past the matrix's last byte become that byte's chunk (those rows' results are
    // never stored)
    const uint8_t *const wsb = a.w + (int64_t)sb * B::BLK;
    const uint32_t ph = (uint32_t)reinterpret_cast<uintptr_t>(wsb) & 15u;
    const uint8_t *const wal = reinterpret_cast<const uint8_t *>(reinterpret_cast<uintptr_t>(wsb) & ~uintptr_t(15));
    const uint32_t rb = (uint32_t)a.row_bytes;
    uint32_t src[NI];
#pragma unroll
    for (int i = 0; i < NI; i++) {
        const int p = min(64 * i + lane, POS - 1);
        const int r = p / CPR, c = p - r * CPR;
        const uint32_t A = ph + (uint32_t)r * rb;
        src[i] = (A & ~15u) + 16u * (uint32_t)min(c, (int)((A & 15u) + B::BLK - 1) >> 4);
    }
    auto issue = [&](int tile, uint8_t *buf) MX_INLINE_LAMBDA {
        const uint8_t *base = wal + (int64_t)tile * MT_ROWS * rb;
        const uint32_t last = (ph + (uint32_t)(min(MT_ROWS, a.n_out - tile * MT_ROWS) - 1) * rb + B::BLK - 1) & ~15u;
#pragma unroll
        for (int i = 0; i < NI; i++) {
            const uint32_t o = min(src[i], last);
            if (64 * (i + 1) <= POS || 64 * i + lane < POS) dma16(base + o, buf + 1024 * i);
        }
        asm volatile("" ::: "memory");
    };
    const uint32_t ph0 = (ph + (uint32_t)n * rb) & 15u;

    // ---- activations: token row n of the group, this wave's super-block ----------
    constexpr int NG = DT == kQ6_K ? 2 : 1;
    half8_t A[8][2];
    {
        const bool on = tok0 + n < a.t;
        const float *xb = a.x + (int64_t)(on ? tok0 + n : 0) * a.k + 256 * sb;
        float v[8][NG][8];
        uint32_t mb = 0;
#pragma unroll
        for (int J = 0; J < 8; J++)
#pragma unroll
            for (int g = 0; g < NG; g++) {
                const float4 *p = reinterpret_cast<const float4 *>(
                    xb + 32 * J + (DT == kQ6_K ? 16 * g + 8 * (q & 1) : 8 * q));
                const float4 u0 = p[0], u1 = p[1];
                const float f[8] = {u0.x, u0.y, u0.z, u0.w, u1.x, u1.y, u1.z, u1.w};
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    v[J][g][i] = on ? f[i] : 0.f;
                    mb = max(mb, __float_as_uint(v[J][g][i]) & 0x7FFFFFFFu);
                }
            }
        mb = max(mb, __float_as_uint(lane_partner<16>(__uint_as_float(mb))));
        mb = max(mb, __float_as_uint(lane_partner<32>(__uint_as_float(mb))));
        // the largest magnitude times 2^-e lies in [2^14, 2^15); a super-block that
        // holds Inf or NaN poisons its token through the scale
        const bool finite = mb < 0x7F800000u, nz = finite && mb != 0;
        int e = nz ? __builtin_amdgcn_frexp_expf(__uint_as_float(mb)) - 15 : 0;
        if (e < -126) e = -126;
        if (q == 0) sTs[wave][n] = !finite ? __builtin_nanf("") : __builtin_amdgcn_ldexpf(1.0f, e);
#pragma unroll
        for (int J = 0; J < 8; J++) {
            float sum = 0.f;
            half8_t h[2], l[2];
#pragma unroll
            for (int g = 0; g < NG; g++)
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    const float f = finite ? __builtin_amdgcn_ldexpf(v[J][g][i], -e) : 0.f;
                    const _Float16 hh = (_Float16)f;
                    h[g][i] = hh;
                    l[g][i] = (_Float16)(f - (float)hh);
                    sum += f;
                }
            if constexpr (DT == kQ6_K) {  // hi in quarters 0, 1, lo of the same values in 2, 3
#pragma unroll
                for (int g = 0; g < 2; g++)
#pragma unroll
                    for (int i = 0; i < 8; i++) A[J][g][i] = q < 2 ? h[g][i] : l[g][i];
            } else {
                A[J][0] = l[0];
                A[J][1] = h[0];
            }
            if constexpr (kMin<DT>) {
                sum += lane_partner<16>(sum);
                sum += lane_partner<32>(sum);
                if (q == 0) sSum[wave][J][n] = sum;
            }
        }
    }
    wait_vmcnt(0);
    wait_lgkmcnt0();
    const float4 ts = *reinterpret_cast<const float4 *>(&sTs[wave][4 * q]);
    int tile = blockIdx.x;
    // (past the last tile: that tile again, so that the copy counts stay exact)
    issue(min(tile, tiles - 1), buf0);
    issue(min(tile + G, tiles - 1), buf1);
    float pend[4];  // finished outputs of the previous tile, stored one stage later
    int prow = -1;
    // outputs tid + 64 W j < 256 of a tile: token 4 (o / 64) + o % 4, row (o / 4) % 16
    auto out = [&](int j, int row0, int64_t &at) MX_INLINE_LAMBDA {
        const int o = tid + 64 * W * j;
        const int tok = tok0 + 4 * (o >> 6) + (o & 3), row = row0 + ((o >> 2) & 15);
        at = (int64_t)tok * a.n_out + row;
        return o < 256 && tok < a.t && row < a.n_out;
    };
    auto flush = [&]() MX_INLINE_LAMBDA {
        if (prow < 0) return;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            int64_t at;
            if (out(j, prow, at)) a.dst[at] = pend[j];
        }
    };
    auto stage = [&](int par, uint8_t *buf) MX_INLINE_LAMBDA {
        wait_vmcnt(NI);  // the stage's copy has landed; the next one's is in flight
        MtW<DT> w;
        w.load(buf + n * SLOT, ph0, q);
        wait_lgkmcnt0();  // the words are in registers: the buffer may be overwritten
        flush();
        issue(min(tile + 2 * G, tiles - 1), buf);
        float4_t sum = {0.f, 0.f, 0.f, 0.f};
        static_for<0, 8>([&](auto jc) MX_INLINE_LAMBDA {
            constexpr int J = decltype(jc)::value;
            const half8_t bf = w.template b<J>();
            if constexpr (DT == kQ6_K) {
                typedef uint32_t u4 __attribute__((ext_vector_type(4)));
                const u4 bw = __builtin_bit_cast(u4, bf);
                u4 g0, g1;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const auto r = __builtin_amdgcn_permlane32_swap(bw[i], bw[i], false, false);
                    g0[i] = r[0];  // the lower half's words in both halves
                    g1[i] = r[1];  // the upper half's
                }
                const float4_t z = {0.f, 0.f, 0.f, 0.f};
                const float4_t d0 =
                    __builtin_amdgcn_mfma_f32_16x16x32_f16(A[J][0], __builtin_bit_cast(half8_t, g0), z, 0, 0, 0);
                const float4_t d1 =
                    __builtin_amdgcn_mfma_f32_16x16x32_f16(A[J][1], __builtin_bit_cast(half8_t, g1), z, 0, 0, 0);
                const float s0 = w.template scale<J, 0>(), s1 = w.template scale<J, 1>();
#pragma unroll
                for (int r = 0; r < 4; r++) sum[r] = __builtin_fmaf(s1, d1[r], __builtin_fmaf(s0, d0[r], sum[r]));
            } else {
                float4_t d = {0.f, 0.f, 0.f, 0.f};
                d = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[J][0], bf, d, 0, 0, 0);
                d = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[J][1], bf, d, 0, 0, 0);
                float s1, c1;
                w.template scales<J>(s1, c1);
#pragma unroll
                for (int r = 0; r < 4; r++) sum[r] = __builtin_fmaf(s1, d[r], sum[r]);
                if constexpr (kMin<DT>) {
                    const float4 sx = *reinterpret_cast<const float4 *>(&sSum[wave][J][4 * q]);
                    sum[0] = __builtin_fmaf(c1, sx.x, sum[0]);
                    sum[1] = __builtin_fmaf(c1, sx.y, sum[1]);
                    sum[2] = __builtin_fmaf(c1, sx.z, sum[2]);
                    sum[3] = __builtin_fmaf(c1, sx.w, sum[3]);
                }
            }
        });
        float f = 1.0f;
        if constexpr (DT == kQ6_K) f = h2f((uint16_t)w.d);
        // (the token's power of two last: f times it may be subnormal, Q6_K with |x| below 2^-113)
        const float4_t acc = {f * sum[0] * ts.x, f * sum[1] * ts.y, f * sum[2] * ts.z, f * sum[3] * ts.w};
        // the waves' partial sums, added in wave order; one barrier a tile (the other
        // parity's buffer is rewritten only after the next tile's barrier)
        *reinterpret_cast<float4_t *>(&sRed[par][wave][4 * lane]) = acc;
        wait_lgkmcnt0();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int o = tid + 64 * W * j;
            float v = 0.f;
            if constexpr (ADD) {  // (the earlier K ranges' sums)
                int64_t at;
                if (out(j, tile * MT_ROWS, at)) v = a.dst[at];
            }
            if (o < 256)
                for (int ww = 0; ww < W; ww++) v += sRed[par][ww][o];
            pend[j] = v;
        }
        prow = tile * MT_ROWS;
        tile += G;
    };
    while (tile < tiles) {  // (block-uniform)
        stage(0, buf0);
        if (tile >= tiles) break;
        stage(1, buf1);
    }
    flush();
    wait_vmcnt(0);  // no copy into this workgroup's LDS outlives it
}

namespace {
template <int DT> void mt_launch(MtArgs a, hipStream_t s) {
    const int nsb = a.k / 256, parts = (nsb + MT_WAVES - 1) / MT_WAVES, per = (nsb + parts - 1) / parts;
    for (a.sb = 0; a.sb < nsb; a.sb += per) {
        const int W = per < nsb - a.sb ? per : nsb - a.sb;
        // resident workgroups: 12 waves per CU by registers, and by LDS
        const int by_lds = 160 * 1024 / (MtLds<DT>::bytes(W) + MtLds<DT>::FIXED), by_waves = MT_WAVES / W;
        const int per_cu = by_lds < by_waves ? by_lds : by_waves;
        const int tiles = (a.n_out + MT_ROWS - 1) / MT_ROWS, most = per_cu * device_cus();
        const dim3 grid((unsigned)(tiles < most ? tiles : most), (unsigned)((a.t + MT_TOK - 1) / MT_TOK));
        if (a.sb) hipLaunchKernelGGL((k_mv_tokens<DT, true>), grid, dim3(64 * W), MtLds<DT>::bytes(W), s, a);
        else hipLaunchKernelGGL((k_mv_tokens<DT, false>), grid, dim3(64 * W), MtLds<DT>::bytes(W), s, a);
    }
}
}  // namespace

// Whether this form is the faster one, from the estimated us of both.  Its launches have a
// latency of their own, one per 12 super-blocks of K, so few rows stay on the per-token
// mat-vecs: Q6_K [512 x 4096], us, per token / here: t = 2 12 / 19, 16 13 / 27; [8192 x
// 4096] t = 2 13 / 24, 8 33 / 27, 16 59 / 32; [100352 x 3072] t = 2 76 / 73, 16 505 / 78;
// Q4_K [8192 x 6144] t = 2 14 / 20, 4 21 / 21, 16 68 / 25.  Rows that the ring kernel does
// not take cost the f32 mat-vec far more per byte: Q4_K at one token [32000 x 7168] 117 /
// 59, [2048 x 14336] 18 / 38.  Of 1370 calls (64 to 100352 rows, K 512 to 28672, 2 to 24
// tokens, replayed in a graph) taking every one here left 292 more than 4% slower than the
// per-token form of before; the line leaves 18, the worst 16% (Q6_K, K 14336).
bool mv_tokens_takes(int dtype, int t, int n_out, int k, int64_t row_bytes) {
    if (t > 65535 * MT_TOK || k <= 0 || k % 256) return false;
    if (t > 65535) return true;  // (the per-token grid's limit)
    const bool ring = mv_ring_fits(dtype, k);
    if (t == 1 && ring) return false;
    // bytes per us and token of the per-token form, bytes per us and pass of this one, us per launch
    struct Rates { double per_token, pass, launch; };
    const Rates r = dtype == kQ4_K   ? Rates{4.0e6, 3.5e6, 8}
                    : dtype == kQ5_K ? Rates{3.5e6, 2.5e6, 8}
                    : dtype == kQ6_K ? Rates{5.5e6, 3.0e6, 10}
                                     : Rates{3.0e6, 2.5e6, 10};
    const double bytes = (double)n_out * (double)row_bytes;
    const int launches = (k / 256 + MT_WAVES - 1) / MT_WAVES, passes = (t + MT_TOK - 1) / MT_TOK;
    const double per_token = 4.0 + t * bytes / (ring ? r.per_token : 1.1e6);
    const double here = launches * r.launch * (1.0 + 0.02 * (t < MT_TOK ? t : MT_TOK)) + passes * bytes / r.pass;
    return here < per_token;
}

mx_status launch_mv_tokens(int dtype, const uint8_t *w, int64_t row_bytes, int n_out, int k, const float *x, int t,
                           float *dst, hipStream_t s) {
    const MtArgs a{w, row_bytes, n_out, k, t, x, dst, 0};
    switch (dtype) {
    case kQ4_K: mt_launch<kQ4_K>(a, s); break;
    case kQ5_K: mt_launch<kQ5_K>(a, s); break;
    case kQ6_K: mt_launch<kQ6_K>(a, s); break;
    default: mt_launch<kQ8_0>(a, s); break;
    }
    MX_LAUNCH("k_mv_tokens");
    return MX_OK;
}

}  // namespace mx
