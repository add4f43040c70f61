// Expert matmuls at a few dozen pairs per expert: activations stationary, weights
// streamed (replaces the kernel_mul_mm_id dispatches, mm_id.metal:492-647, at
// these sizes).
//
// At such sizes the launch is a stream of weights, and what bounds a tile that
// walks K in small steps over many rows (the grouped GEMM: 64 quant bytes of each
// of 512 rows a step) is the access pattern: every 128-byte line is fetched about
// 1.6 times and a copy instruction touches some 20 lines.  Here a workgroup reads
// whole rows: its W waves split K, each owning NSB super-blocks (256 values) and
// holding the f16 activations of a run of 16 * MT pairs for them in registers as
// MFMA operands; it walks 16-row tiles of the expert's matrix, each wave
// contracting its K share (v_mfma_f32_16x16x32_f16), and the waves' partial sums
// meet in LDS in wave order.  Weights are dequantised as in the verify tiles and
// the grouped GEMM (the f16 rounding of the f32 value, mx_wb.h); A rows are f16
// times a power of two per row; sums are f32.
//
//  * Which launches: those with few runs for their m-tiles of 128 pairs, decided from
//    the map by every workgroup alike (gs_ratio); the grouped GEMM launched next reads
//    the answer and leaves or does the work.
//  * Work: the runs of all experts (each expert's bucket cut into 16 * MT pairs)
//    times the row tiles, cut into one contiguous share per resident workgroup:
//    a workgroup loads a run's activations once per share and run.  The map gives
//    the pairs per expert; every workgroup forms the prefix of the runs itself.
//  * Copies: two stage buffers per wave (16 rows x one super-block, the 16-byte
//    chunks that cover it); the copy of the stage after the next is issued as soon
//    as a stage's words are in registers, across tiles and runs.
//  * Short K: several teams of waves per workgroup, each on its own tiles of the run,
//    so that a CU holds 12 waves of one super-block (168 registers) or 8 of more.
//  * SwiGLU: a tile is 16 gate rows, then the same 16 up rows; the thread that
//    sums a gate value keeps it until its up value is summed.
//
// Bound by instruction issue and the waits between: about 170 (Q4_K) to 250 (Q6_K) VALU per
// wave and stage of 16 x 256 weights, once per run of 32 pairs; VALU and MFMA instructions
// execute in 64 to 70% of the SIMD cycles.  top-10 of 256 experts, hidden 4096,
// ff 1536, Q4_K / Q6_K, grouped GEMM against these (gate, up and down with the
// passes between them): t = 300 1180 / 892 us, 512 1267 / 1078, 700 1410 / 1300,
// 1000 1548 / 1590.  Weight bytes fetched for the gate projection at t = 512: 1.46 ->
// 1.19 GB (0.91 GB of weights, read once per run).  Also tried: reading a stage's
// words one stage ahead (no change: latency of LDS is not what it waits on), and the
// grouped GEMM's tiles with three weight buffers and only the A rows that exist
// (1279 -> 1420 us).
#include "mx_launch.h"
#include "mx_dma.h"
#include "mx_wb.h"
#include "mx_vmq.h"

namespace mx {

namespace {

constexpr int GS_MAX_E = 1025;  // map experts (routed and shared)

// per type: super-block bytes, 16-byte chunks copied per row (slots as long: 16 rows on distinct banks)
template <int DT> struct GsBlk;
template <> struct GsBlk<kQ4_K> { static constexpr int BLK = 144, CPR = 9; };
template <> struct GsBlk<kQ5_K> { static constexpr int BLK = 176, CPR = 11; };
template <> struct GsBlk<kQ6_K> { static constexpr int BLK = 210, CPR = 15; };
template <> struct GsBlk<kQ8_0> { static constexpr int BLK = 272, CPR = 19; };

// half super-block PAR of the lane's row from its slot (ph: the block's phase)
template <int PAR> __device__ __forceinline__ void gs_load(VmQ4 &w, const uint8_t *slot, int q, uint32_t) {
    w.template load<PAR>(slot, q);
}
template <int PAR> __device__ __forceinline__ void gs_load(WB<kQ5_K> &w, const uint8_t *slot, int q, uint32_t) {
    const int kh = q >> 1;
    w.h = ld_w4(slot);
    w.qh = ld_w4(slot + 16 + 16 * kh);
    w.q[0] = ld_w4(slot + 48 + 64 * PAR + 16 * kh);
    w.q[1] = ld_w4(slot + 80 + 64 * PAR + 16 * kh);
}
template <int PAR> __device__ __forceinline__ void gs_load(VmQ6 &w, const uint8_t *slot, int q, uint32_t ph) {
    w.template load<PAR>(slot, q, ph);
}
template <int PAR> __device__ __forceinline__ void gs_load(WB<kQ8_0> &w, const uint8_t *slot, int q, uint32_t ph) {
    w.load_lds(slot, q >> 1, ph + 136 * PAR, 0);
}

// Ten times the most runs per m-tile of the map at which a launch is taken.  The
// average of pairs per expert, all the host knows, does not tell: with a router that
// uses a quarter of 256 experts (hidden 4096, ff 1536, Q4_K / Q6_K) 12 pairs on average
// took 414 us in the grouped GEMM and 461 here, 20: 485 / 662; evenly used experts of 24
// pairs 290 / 239, of 40 (1.9 runs per m-tile) 299 / 304.  By type, from even use: plain
// [4096 x 1536] Q5_K of 24 pairs 122 / 115, 36: 130 / 142; Q6_K 36: 185 / 145; Q8_0 24:
// 146 / 147; SwiGLU hidden 3072 Q6_K of 40: 482 / 392, Q8_0 440 / 463.
__host__ __device__ constexpr int gs_ratio(int dtype, bool swiglu) {
    return dtype == kQ6_K ? (swiglu ? 22 : 18) : dtype == kQ4_K ? 16 : swiglu ? 15 : 13;
}

// Gate/up of the cheaply unpacked types are taken below 40 * fill - 14 pairs per m-tile, fill:
// the share of the CU's waves and super-blocks that K fills (9 at K = 1792, 26 where all are).
// A stage costs a run the same whatever its pairs, and few waves make every stage slower,
// while the GEMM gains with the pairs.  Layers, time here over the GEMM's (or the tiles'),
// even routers, at 8 / 16 / 24 pairs per expert: Q4_K K = 1536 0.91 / 0.98 / 1.02, 1792 0.99 /
// 1.06 / 1.13, 2048 at 16 / 24 1.04 / 1.10, 3072 0.96 / 0.88 / 0.97; Q5_K 1792 0.97 / 1.05 / 1.07,
// 3584 1.00 / 1.03 / 1.08; Q6_K 1792 0.85 / 0.86 / 0.94 (no line).
__host__ __device__ constexpr bool gs_by_fill(int dtype, bool swiglu) { return swiglu && dtype != kQ6_K; }

template <int DT, bool SWIGLU, int MT, int NSB, int WM> struct GsGeo {
    static constexpr int CPR = GsBlk<DT>::CPR, BLK = GsBlk<DT>::BLK, SLOT = 16 * CPR;
    static constexpr int POS = 16 * CPR, NI = (POS + 63) / 64, STAGE = POS * 16;
    // waves of a workgroup at most: teams of at most WM waves
    static constexpr int WAVES = NSB == 1 ? 12 : 8;
    // waves per SIMD the registers must allow: 3 (168) for one super-block, else 2
    static constexpr int WPE = NSB == 1 ? 3 : 2;
    static constexpr int OUT = MT * 256;             // sums per tile and matrix
    // finished sums per thread: a team has at least WMIN waves
    static constexpr int WMIN = WM == 12 ? 7 : WM == 8 ? (NSB > 2 ? 6 : 7) : WM == 6 ? 5 : WM == 4 ? 3 : 2;
    static constexpr int TEAMS = WAVES / WMIN;  // teams at most
    static constexpr int FIXED = (2 * TEAMS * WM * OUT + GS_MAX_E + 1 + WAVES + 4 * 16 * MT) * 4;  // static LDS
    static constexpr int JM = (OUT + 64 * WMIN - 1) / (64 * WMIN);
};

}  // namespace

template <int DT, bool SWIGLU, int MT, int NSB, int WM>
__global__ void __launch_bounds__((64 * GsGeo<DT, SWIGLU, MT, NSB, WM>::WAVES))
    __attribute__((amdgpu_waves_per_eu(GsGeo<DT, SWIGLU, MT, NSB, WM>::WPE)))
k_gst(GemmArgs a, int W) {
    using G = GsGeo<DT, SWIGLU, MT, NSB, WM>;
    using WT = std::conditional_t<DT == kQ4_K, VmQ4, std::conditional_t<DT == kQ6_K, VmQ6, WB<DT>>>;
    constexpr int NI = G::NI, POS = G::POS, CPR = G::CPR, BLK = G::BLK, RUN = 16 * MT, OUT = G::OUT;
    constexpr int NMAT = SWIGLU ? 2 : 1;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];  // the stage buffers, two per wave
    // partial sums, two parities (rows of a team past its waves stay zero)
    constexpr int TEAMS = G::TEAMS;
    __shared__ __attribute__((aligned(16))) float sRed[2][TEAMS][WM][OUT];
    __shared__ int sRuns[GS_MAX_E + 1];  // runs before expert e
    __shared__ int sScan[G::WAVES];
    __shared__ int sOutRow[2][RUN];
    __shared__ float sScale[2][RUN];
    const int tid = threadIdx.x, lane = tid & 63;
    // teams of W waves (one super-block range per wave of a team); a team takes every
    // teams-th tile of a run
    const int gwave = __builtin_amdgcn_readfirstlane(tid >> 6), teams = (int)(blockDim.x >> 6) / W;
    const int team = gwave / W, wave = gwave - team * W;
    const int NT = 64 * W, ttid = 64 * wave + (tid & 63), BT = blockDim.x;
    const int n = lane & 15, q = lane >> 4, hh = q & 1, kh = q >> 1;
    const int E = a.n_map_expert;
    const MapLayout L(E, a.t, a.top_k);

    // ---- the runs of every expert: exclusive prefix ---------------------------------
    int runs;
    {
        const int per = (E + BT - 1) / BT, e0 = min(tid * per, E), e1 = min(e0 + per, E);
        int sum = 0;  // runs, and m-tiles of 128 pairs in the upper half (both below 2^15: gst_fits)
        for (int e = e0; e < e1; e++) {
            const int v = a.map[L.tpe + e];
            sum += (v + RUN - 1) / RUN + ((v + GM_BM - 1) / GM_BM << 16);
        }
        int inc = sum;  // inclusive scan over the wave's lanes
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int v = __shfl_up(inc, d);
            if (lane >= d) inc += v;
        }
        if (lane == 63) sScan[gwave] = inc;
        __syncthreads();
        int base = inc - sum, both = 0;
        for (int w = 0; w < W * teams; w++) {
            const int v = sScan[w];
            both += v;
            if (w < gwave) base += v;
        }
        both = __builtin_amdgcn_readfirstlane(both);
        // many runs for their m-tiles: the grouped GEMM is the faster (block-uniform; nothing
        // else is done before this: a launch left behind costs 2 to 2.5 us)
        runs = both & 0xFFFF;
        const int mtiles = both >> 16, fill = 40 * (a.k / 256) * teams / (G::WAVES * NSB) - 14;
        const bool mine = 10 * runs < gs_ratio(DT, SWIGLU) * mtiles &&
                          (!gs_by_fill(DT, SWIGLU) || a.t * a.top_k < fill * mtiles);
        if (blockIdx.x == 0 && tid == 0) *a.done = mine;
        if (!mine) return;
        for (int e = e0; e < e1; e++) {
            sRuns[e] = base & 0xFFFF;
            base += (a.map[L.tpe + e] + RUN - 1) / RUN;
        }
        if (tid == 0) sRuns[E] = runs;
        for (int i = tid; i < 2 * TEAMS * WM * OUT; i += BT) (&sRed[0][0][0][0])[i] = 0.f;
        __syncthreads();
    }
    const int tiles = a.n_out / 16;
    // this workgroup's share [u0, u1) of the runs * tiles units; neighbouring shares on
    // one XCD (workgroups are dealt to the 8 XCDs round-robin)
    const int64_t total = (int64_t)runs * tiles;
    const int nwg = (int)gridDim.x, c = (blockIdx.x & 7) * (nwg >> 3) + (blockIdx.x >> 3);
    const int64_t u0 = total * c / nwg, u1 = total * (c + 1) / nwg;
    if (u0 >= u1) return;  // (block-uniform)
    const int nsb = a.k / 256, sb0 = wave * NSB, cnt = min(NSB, nsb - sb0);  // >= 1
    // passes of `teams` tiles: a run's tiles of the share, run by run
    const int run0 = (int)(u0 / tiles), run1 = (int)((u1 - 1) / tiles);
    const int first = (int)(u0 - (int64_t)run0 * tiles), last = (int)(u1 - (int64_t)run1 * tiles);
    auto end_of = [&](int r) { return r == run1 ? last : tiles; };
    int64_t passes = 0;
    {
        auto up = [&](int v) { return (v + teams - 1) / teams; };
        if (run0 == run1) passes = up(last - first);
        else passes = up(tiles - first) + (int64_t)(run1 - run0 - 1) * up(tiles) + up(last);
    }
    const int64_t stages = passes * NMAT * cnt;

    // the expert of run r (block-uniform)
    auto expert_of = [&](int r) {
        int lo = 0, hi = E;  // sRuns[lo] <= r < sRuns[hi]
        while (hi - lo > 1) {
            const int m = (lo + hi) >> 1;
            if (sRuns[m] <= r) lo = m;
            else hi = m;
        }
        return __builtin_amdgcn_readfirstlane(lo);
    };

    // ---- copies: a cursor of its own, two stages ahead of the contraction --------------
    uint8_t *const buf0 = lds + gwave * (2 * G::STAGE), *const buf1 = buf0 + G::STAGE;
    const uint32_t rb = (uint32_t)(a.row_bytes);  // (the shared expert's rows have the same width)
    uint32_t src[NI];  // the lane's chunks from the tile's first byte, for super-block sb0
    // a tile starts 16-byte aligned; block (row, sb) at row * rb + sb * BLK
    auto chunk = [&](int i, int sb) MX_INLINE_LAMBDA {
        const int p = min(64 * i + lane, POS - 1);
        const int r = p / CPR, cc = p - r * CPR;
        const uint32_t A = (uint32_t)r * rb + (uint32_t)(sb * BLK);
        return (A & ~15u) + 16u * (uint32_t)min(cc, (int)((A & 15u) + BLK - 1) >> 4);
    };
#pragma unroll
    for (int i = 0; i < NI; i++) src[i] = chunk(i, sb0);
    int i_run = run0, i_tile = first, i_end = end_of(run0), i_mat = 0, i_s = 0;
    const uint8_t *i_w[NMAT];
    auto matrices = [&](int r) MX_INLINE_LAMBDA {
        const int e = expert_of(r);
        const bool sh = e >= a.n_expert;
#pragma unroll
        for (int m = 0; m < NMAT; m++) i_w[m] = sh ? a.w_sh[m] : a.w[m] + (int64_t)e * a.expert_bytes;
    };
    matrices(i_run);
    int64_t left = stages;  // stages not yet issued
    auto issue = [&](uint8_t *buf) MX_INLINE_LAMBDA {
        const uint8_t *base = (NMAT == 2 && i_mat ? i_w[NMAT - 1] : i_w[0]) + (int64_t)min(i_tile + team, i_end - 1) * 16 * rb;
#pragma unroll
        for (int i = 0; i < NI; i++) {
            uint32_t o = src[i];
            if constexpr (NSB > 1) {
                if constexpr (DT == kQ6_K) o = i_s ? chunk(i, sb0 + i_s) : o;  // (another phase)
                else o += (uint32_t)(i_s * BLK);
            }
            if (64 * (i + 1) <= POS || 64 * i + lane < POS) dma16(base + o, buf + 1024 * i);
        }
        asm volatile("" ::: "memory");
        // the next stage (past the last one: it again, so that the counts stay exact)
        if (--left <= 0) return;
        if (++i_s < cnt) return;
        i_s = 0;
        if (++i_mat < NMAT) return;
        i_mat = 0;
        if ((i_tile += teams) < i_end) return;
        i_tile = 0;
        matrices(++i_run);
        i_end = end_of(i_run);
    };

    // ---- contraction ---------------------------------------------------------------
    half8_t A[NSB][MT][8];
    int run = run0, tile = first, tab = 0;
    auto load_run = [&]() MX_INLINE_LAMBDA {
        const int e = expert_of(run);
        const int pos0 = a.map[L.off + e] + (run - sRuns[e]) * RUN;
        const int rows = min(RUN, a.map[L.off + e] + a.map[L.tpe + e] - pos0);
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
            const int m = min(16 * mt + n, rows - 1);  // missing pairs repeat the last: never stored
            const int pos = pos0 + m;
            const int64_t ar = a.a_div ? a.map[L.list + pos] / a.a_div : pos;
            const _Float16 *ap = a.a + ar * a.k;
#pragma unroll
            for (int s = 0; s < NSB; s++) {
                const _Float16 *p = ap + (sb0 + min(s, cnt - 1)) * 256 + (DT == kQ4_K ? 32 : 8) * q;
#pragma unroll
                for (int i = 0; i < 8; i++)
                    A[s][mt][i] = *reinterpret_cast<const half8_t *>(p + 128 * (i >> 2) + (DT == kQ4_K ? 8 : 32) * (i & 3));
            }
        }
        // the rows have landed (used later, next to copies in flight that the compiler
        // would wait for with them)
        wait_vmcnt(0);
#pragma unroll
        for (int s = 0; s < NSB; s++)
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    asm volatile("" : "+v"(A[s][mt][i]));
                    // (VmQ4's weights come in the order 0, 2, 1, 3 of each four)
                    if constexpr (DT == kQ4_K)
                        A[s][mt][i] = __builtin_shufflevector(A[s][mt][i], A[s][mt][i], 0, 2, 1, 3, 4, 6, 5, 7);
                }
        tab ^= 1;
        for (int m = tid; m < RUN; m += BT) {
            const int pos = pos0 + min(m, rows - 1);
            const int pair = a.map[L.list + pos];
            sScale[tab][m] = a.a_scale[a.a_div ? pair / a.a_div : pos];
            sOutRow[tab][m] = m >= rows ? -1 : SWIGLU ? pos : pair / a.top_k * a.out_stride + pair % a.top_k + a.out_add;
        }
    };
    issue(buf0);
    issue(buf1);
    load_run();
    // finished sums o = ttid + NT j < OUT of a tile: pair 16 (o / 256) + 4 (o / 64 % 4) + o % 4, row o / 4 % 16
    constexpr int JM = G::JM;
    float pend[JM], gate[JM];
    int prow[JM];
#pragma unroll
    for (int j = 0; j < JM; j++) prow[j] = -1;
    int pcol = 0;
    auto flush = [&]() MX_INLINE_LAMBDA {
#pragma unroll
        for (int j = 0; j < JM; j++)
            if (prow[j] >= 0) a.out[(int64_t)prow[j] * a.n_out + pcol + ((ttid + NT * j) >> 2 & 15)] = pend[j];
#pragma unroll
        for (int j = 0; j < JM; j++) prow[j] = -1;
    };
    float4_t acc[MT];
    int mat = 0, par = 0, t_end = end_of(run0);
    // one pass: this tile's rows of matrix `mat`, the wave's super-blocks; odd: the
    // first stage is in buf1
    int odd = 0;
    for (;;) {
#pragma unroll
        for (int mt = 0; mt < MT; mt++) acc[mt] = float4_t{0.f, 0.f, 0.f, 0.f};
        static_for<0, NSB>([&](auto sc) MX_INLINE_LAMBDA {
            constexpr int s = decltype(sc)::value;
            if (s < cnt) {  // wave-uniform
                uint8_t *const buf = odd ? buf1 : buf0;
                odd ^= 1;
                wait_vmcnt(NI);  // the stage's copy has landed; the next one's is in flight
                const uint8_t *slot = buf + n * G::SLOT;
                const uint32_t ph = ((uint32_t)n * rb + (uint32_t)((sb0 + s) * BLK)) & 15u;
                WT w0, w1;
                gs_load<0>(w0, slot, q, ph);
                gs_load<1>(w1, slot, q, ph);
                wait_lgkmcnt0();  // the words are in registers: the buffer may be overwritten
                if (s == 0) flush();
                issue(buf);
                auto half = [&](auto parc, WT &w) MX_INLINE_LAMBDA {
                    constexpr int PAR = decltype(parc)::value;
                    if constexpr (DT == kQ6_K) w.prep(kh);
                    else if constexpr (DT != kQ4_K) w.template prep<PAR>(kh);
                    static_for<0, 4>([&](auto pc) MX_INLINE_LAMBDA {
                        constexpr int P = decltype(pc)::value;
                        half8_t bf;
                        if constexpr (DT == kQ4_K) bf = w.step(P);
                        else if constexpr (DT == kQ6_K) bf = w.template step<P>();
                        else bf = w.step(P, hh);
#pragma unroll
                        for (int mt = 0; mt < MT; mt++)
                            acc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[s][mt][4 * PAR + P], bf, acc[mt], 0, 0, 0);
                    });
                };
                half(std::integral_constant<int, 0>{}, w0);
                half(std::integral_constant<int, 1>{}, w1);
            }
        });
#pragma unroll
        for (int mt = 0; mt < MT; mt++) *reinterpret_cast<float4_t *>(&sRed[par][team][wave][256 * mt + 4 * lane]) = acc[mt];
        wait_lgkmcnt0();
        __builtin_amdgcn_s_barrier();  // (one a pass: the other parity is rewritten only after the next)
        asm volatile("" ::: "memory");
#pragma unroll
        for (int j = 0; j < JM; j++) {
            const int o = ttid + NT * j;
            if (o < OUT) {
                float v = 0.f;
#pragma unroll
                for (int w = 0; w < WM; w++) v += sRed[par][team][w][o];
                const int m = 16 * (o >> 8) + 4 * ((o >> 6) & 3) + (o & 3);
                v *= sScale[tab][m];
                if (SWIGLU && mat == 0) gate[j] = v;
                else {
                    // silu(g) * u on the hardware exp2 and reciprocal, as the grouped GEMM
                    if constexpr (SWIGLU)
                        v = gate[j] * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-gate[j] * 1.4426950408889634f)) * v;
                    pend[j] = v;
                    prow[j] = tile + team < t_end ? sOutRow[tab][m] : -1;
                }
            }
        }
        par ^= 1;
        if (++mat < NMAT) continue;
        mat = 0;
        pcol = (tile + team) * 16;
        if ((tile += teams) < t_end) continue;
        if (run == run1) break;
        tile = 0;
        t_end = end_of(++run);
        flush();
        load_run();
    }
    flush();
    wait_vmcnt(0);  // no copy into this workgroup's LDS outlives it
}

namespace {
template <int DT, bool SWIGLU, int MT, int NSB, int WM> void gs_go(const GemmArgs &a, hipStream_t s) {
    using G = GsGeo<DT, SWIGLU, MT, NSB, WM>;
    const int W = (a.k / 256 + NSB - 1) / NSB, teams = G::WAVES / W;
    static_assert(G::FIXED + G::WAVES * 2 * G::STAGE <= 160 * 1024, "one workgroup per CU");
    // one workgroup per CU, a multiple of 8: one group of shares per XCD
    const unsigned grid = (unsigned)(device_cus() & ~7);
    hipLaunchKernelGGL((k_gst<DT, SWIGLU, MT, NSB, WM>), dim3(grid), dim3(64 * W * teams), W * teams * 2 * G::STAGE, s, a, W);
}
// pairs per run of the instantiation gs_launch takes
int gs_run(int dtype, bool swiglu, int nsb) { return nsb > 16 || (dtype == kQ8_0 && !swiglu && nsb <= 4) ? 16 : 32; }
// W waves of NSB super-blocks: all the super-blocks of a run's pairs fit the CU's
// registers (12 waves of one, 8 of more), in several teams where K is short
template <int DT, bool SWIGLU> void gs_launch(const GemmArgs &a, hipStream_t s) {
    const int nsb = a.k / 256;
    if constexpr (DT == kQ8_0) {  // (its raw words spill at 168 registers next to two pair tiles)
        if constexpr (!SWIGLU) {  // (gst_fits)
            if (nsb <= 2) return gs_go<DT, SWIGLU, 1, 1, 2>(a, s);
            if (nsb <= 4) return gs_go<DT, SWIGLU, 1, 1, 4>(a, s);
        }
        if (nsb <= 8) return gs_go<DT, SWIGLU, 2, 2, 4>(a, s);
        if (nsb <= 12) return gs_go<DT, SWIGLU, 2, 2, 6>(a, s);
    } else {
        if constexpr (!SWIGLU) {
            if (nsb <= 2) return gs_go<DT, SWIGLU, 2, 1, 2>(a, s);
            if (nsb <= 4) return gs_go<DT, SWIGLU, 2, 1, 4>(a, s);
        }
        if (nsb <= 6) return gs_go<DT, SWIGLU, 2, 1, 6>(a, s);
        if (nsb <= 12) return gs_go<DT, SWIGLU, 2, 1, 12>(a, s);
    }
    if (nsb <= 16) return gs_go<DT, SWIGLU, 2, 2, 8>(a, s);
    if (nsb <= 24) return gs_go<DT, SWIGLU, 1, 3, 8>(a, s);
    gs_go<DT, SWIGLU, 1, 4, 8>(a, s);
}
}  // namespace

bool gst_fits(int dtype, const GemmArgs &a, bool swiglu) {
    auto al = [](const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    const bool sh = a.w_sh[0] != nullptr;
    bool ok = a.k % 256 == 0 && a.k / 256 >= 2 && a.k / 256 <= 32 && a.n_out % 16 == 0 && a.n_map_expert < GS_MAX_E &&
              a.row_bytes < (1 << 24) && (!sh || a.sh_row_bytes == a.row_bytes);
    for (int m = 0; m < (swiglu ? 2 : 1); m++)
        ok = ok && (a.n_expert == 0 || (al(a.w[m]) && a.expert_bytes % 16 == 0)) && (!sh || al(a.w_sh[m]));
    // Gate/up of K up to 1024 stay on the grouped GEMM: a layer of hidden 1024, ff 512, 64
    // experts, Q6_K / Q4_K, took 92 us there, 101 with both projections here and 96 with the down alone (28 pairs).
    ok = ok && (!swiglu || a.k > 1024);
    // Matrices of at least 256 MB in all (what the Infinity Cache holds): below, the grouped
    // GEMM's repeated reads are cheap, and the launch left behind under a skewed router is a
    // larger share of the layer (layers, us, the GEMM alone / here: hidden 1024, ff 512, 64
    // experts Q5_K 62 / 71; hidden 2048, ff 768, 128 experts Q4_K / Q6_K at 200 tokens, even
    // router 206 / 180, skewed 115 / 122).  Smaller ones where the GEMM has too little to run
    // on, up to 12 pairs per expert and half a workgroup per CU (60 random layers 0.90 of its
    // time, 7 more than 4% slower), and Q6_K gate/up, which the GEMM unpacks slowest (73 layers
    // 0.90, 2 slower; hidden 3584, ff 256, 16 experts at 40 tokens 110 / 60).
    const int64_t bytes = (int64_t)a.n_map_expert * a.n_out * a.row_bytes * (swiglu ? 2 : 1);
    const int rows = swiglu ? 2 * a.n_out : a.n_out, wg = !swiglu && (dtype == kQ6_K || dtype == kQ8_0) ? 256 : 512;
    const bool idle = 2 * (int64_t)a.n_map_expert * ((rows + wg - 1) / wg) <= device_cus() &&
                      (int64_t)a.t * a.top_k < 12 * (int64_t)a.n_map_expert;
    ok = ok && (bytes >= (int64_t)256 << 20 || idle || (swiglu && dtype == kQ6_K));
    // Less than one run per expert on average: beyond, even an evenly used map has two runs
    // per m-tile, which no gs_ratio takes where runs are of 16 pairs and few do at 32; what it
    // takes gained 1.08 (27 pairs) to 1.3x (12 pairs).
    return ok && (int64_t)a.t * a.top_k < gs_run(dtype, swiglu, a.k / 256) * (int64_t)a.n_map_expert;
}

mx_status launch_gst(int dtype, bool swiglu, const GemmArgs &a, hipStream_t s) {
    if (a.t == 0) return MX_OK;
#define MX_P(DT) if (swiglu) gs_launch<DT, true>(a, s); else gs_launch<DT, false>(a, s)
    switch (dtype) {
    case kQ4_K: MX_P(kQ4_K); break;
    case kQ5_K: MX_P(kQ5_K); break;
    case kQ6_K: MX_P(kQ6_K); break;
    default: MX_P(kQ8_0); break;
    }
#undef MX_P
    MX_LAUNCH("k_gst");
    return MX_OK;
}

}  // namespace mx
