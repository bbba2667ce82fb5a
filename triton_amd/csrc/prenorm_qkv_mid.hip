// Fused RMSNorm + Q/K/V projection for problems between the weight stream of a few tokens (prenorm_qkv_skinny.hip) and
// the tilings that fill the chip by themselves (prenorm_qkv.hip, prenorm_qkv_wide.hip): some 33 to 700 tokens at the
// Llama3-8B widths.
//
// What bounds it: a 128-column tile of a 4096-deep projection is 64 k-tiles in sequence, and with at most one tile per
// CU each costs the latency of its weights from HBM -- 1.1 us with the two stages of the 128 x 128 kernel, whatever the
// token count (70 us from 33 to 600 tokens).  Hence a ring of four stages of 64 contraction columns, filled by direct
// global->LDS loads with whole 128-byte lines of both operands, and tiles small enough to occupy the CUs: 64 or 128
// tokens x 64 columns while those do not exceed one per CU, then 128 x 128.  Deeper rings lose: the weights' row pitch
// is a power of two at these widths, the panels of a row share its DRAM pages, and every extra stage in flight pulls the
// workgroups further apart along the contraction (eight W stages: 39 -> 45 us).
//
// The eight waves are TM token groups x TN column groups x four contraction steps of 16: a wave owns 32 NTB tokens x 64
// columns of its stage's 16-column step, so that its operands feed 2 NTB MFMAs each stage, and the four partial tiles
// are added through LDS at the end.  One barrier per stage; the operands of the next stage are read behind the MFMAs of
// the one in hand.  gamma is multiplied into the X operand, NTB products a stage instead of two: gamma * w falls out of the
// normal fp16 range where gamma * x does not (distance from float64 with gamma around 1e-3 and weights of 0.02: 8.9e-4
// against 2.9e-4).  The sum of squares is taken from X as read, by the waves of the first column group.
//
// Measured, weights cold in HBM, us before (128 x 128 kernel) / now: 4096 -> 12288 without norm 33 tokens 63 / 26, 64
// tokens 63 / 29, 100 tokens 64 / 35; 4096 -> 6144 with norm and gamma 100 tokens 74 / 26, 256 tokens 74 / 37.5, 512 tokens
// 74 / 43; 1024 -> 3072 128 tokens 18 / 8.
#include "prenorm_qkv.h"

namespace trn {

template <int NTB, int TM, int TN, int NORM, bool STREAM>      // NORM: 0 none, 1 without gamma, 2 with gamma; STREAM: W past the caches
__global__ __launch_bounds__(512, 2) void prenorm_qkv_mid_kernel(const GemmArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)   // buffer descriptors and LDS-load builtins exist in the device pass only
    static_assert(TM * TN == 2, "eight waves: two tiles x four contraction steps");
    constexpr int KQ = 4, NW = 8, MT = TM * NTB * 32, NT = TN * 64, SK = 64;
    constexpr int XI = MT / 8 / NW, WI = NT / 8 / NW, NL = XI + WI + (NORM == 2 ? 1 : 0);    // requests of a stage per wave
    // One array per stage: the compiler orders LDS reads after outstanding global->LDS loads that may alias them, and
    // only distinct variables are provably disjoint.
    __shared__ __attribute__((aligned(1024))) half_t S0[(MT + NT) * SK];
    __shared__ __attribute__((aligned(1024))) half_t S1[(MT + NT) * SK];
    __shared__ __attribute__((aligned(1024))) half_t S2[(MT + NT) * SK];
    __shared__ __attribute__((aligned(1024))) half_t S3[(MT + NT) * SK];
    __shared__ float ss_part[KQ][MT];

    const int tid = threadIdx.x, lane = tid & 63, c = lane & 31, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kq = wave % KQ, tn = wave / KQ % TN, tm = wave / (KQ * TN);
    // Workgroup ids are dealt round-robin to the 8 XCDs: the token tiles of a panel share one XCD's L2, neighbouring
    // panels sit on different ones.
    const int mt = (blockIdx.x >> 3) % a.n_mtiles, panel = (blockIdx.x & 7) + 8 * ((blockIdx.x >> 3) / a.n_mtiles);
    if (panel >= a.n_panels) return;
    const int pi = panel >= a.p[2].tile0 ? 2 : (panel >= a.p[1].tile0 ? 1 : 0);
    const ProjOut P = a.p[pi];
    const int n0 = (panel - P.tile0) * NT, m0 = mt * MT;
    const int nst = (a.K + SK - 1) / SK;
    constexpr int kOut = 0x7ffffff0;                 // a byte offset past every buffer: the load returns zeros

    // ---- W stage: TN groups of [64 rows][64 columns], chunk c of row r at c ^ swz<64>(r).  A wave-wide load covers 8 rows.
    const __amdgpu_buffer_rsrc_t wrs = __builtin_amdgcn_make_buffer_rsrc(
        (void*)P.w, 0, (int)(((int64_t)(a.K - 1) * P.ldw + P.n) * 2), 0x00020000);
    int w_vo[WI];
#pragma unroll
    for (int i = 0; i < WI; ++i) {
        const int j = wave * WI + i, r = 8 * (j & 7) + (lane >> 3);
        w_vo[i] = (int)(r * P.ldw * 2) + (n0 + (j >> 3) * 64 + 8 * ((lane & 7) ^ swz<64>(r))) * 2;
    }
    const int w_stage = (int)(SK * P.ldw * 2);
    // ---- X stage: [MT tokens][64 columns], chunk c of row r at c ^ ((r/2) % 8) (128-byte rows: two share a line of the
    // 64 banks, and the 16 lanes of a read that are served together hold each (row parity, slot) once)
    const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc(
        (void*)a.x, 0, (int)(((int64_t)(a.T - 1) * a.ldx + a.K) * 2), 0x00020000);
    int x_vo[XI], x_ch[XI];
#pragma unroll
    for (int i = 0; i < XI; ++i) {
        const int r = 8 * (XI * wave + i) + (lane >> 3), t = m0 + r;
        x_ch[i] = (lane & 7) ^ ((r >> 1) & 7);
        x_vo[i] = t < a.T ? (int)(t * a.ldx * 2) + x_ch[i] * 16 : kOut;          // rows past the end read as zeros
    }
    // ---- gamma: the 16 columns of this wave's contraction step, a register ring like the stages
    const __amdgpu_buffer_rsrc_t grs = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(NORM == 2 ? a.gamma : a.x), 0, NORM == 2 ? a.K * 2 : 0, 0x00020000);
    half8_t g0, g1, g2, g3;
    // Request n of a stage's NL (gamma, W, X); past the last stage they read rows past hidden, i.e. zeros.
    auto request = [&](int n, int s, half_t* D, half8_t& g) __attribute__((always_inline)) {
        const int st = min(s, nst), i = n - (NL - XI - WI);
        if (i < 0)
            g = __builtin_bit_cast(half8_t, __builtin_amdgcn_raw_buffer_load_b128(grs, (kq * 16 + 8 * h) * 2, st * SK * 2, 0));
        else if (i < WI)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                wrs, (__attribute__((address_space(3))) void*)(D + MT * SK + (wave * WI + i) * 512), 16, w_vo[i], st * w_stage, 0, STREAM ? 2 : 0);
        else              // columns past hidden hold the next row's data: read zeros instead
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                xrs, (__attribute__((address_space(3))) void*)(D + (XI * wave + i - WI) * 512), 16,
                st * SK + 8 * x_ch[i - WI] >= a.K ? kOut : x_vo[i - WI], st * SK * 2, 0, 0);
    };
    auto fetch = [&](int s, half_t* D, half8_t& g) __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int n = 0; n < NL; ++n) request(n, s, D, g);
        __builtin_amdgcn_sched_barrier(0);
    };

    // ---- LDS read offsets (halfs) within a stage: W^T A-operand through the transposing read, X^T B-operand
    int woff_lo[2], woff_hi[2], xoff[NTB];
    {
        const int rl = 8 * h + ((lane & 15) >> 2), rh = rl + 4;
        const int lc = 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1), sub = (lane & 1) * 4;
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) {
            woff_lo[nb] = MT * SK + tn * 4096 + (kq * 16 + rl) * 64 + (((nb * 4 + lc) ^ swz<64>(rl)) << 3) + sub;
            woff_hi[nb] = MT * SK + tn * 4096 + (kq * 16 + rh) * 64 + (((nb * 4 + lc) ^ swz<64>(rh)) << 3) + sub;
        }
#pragma unroll
        for (int tb = 0; tb < NTB; ++tb) {
            const int r = (tm * NTB + tb) * 32 + c;
            xoff[tb] = r * SK + (((2 * kq + h) ^ ((r >> 1) & 7)) << 3);
        }
    }
    auto read_w = [&](const half_t* C, int nb) __attribute__((always_inline)) {
        const half4_t lo = lds_read_tr16(C + woff_lo[nb]);
        const half4_t hi = lds_read_tr16(C + woff_hi[nb]);
        return half8_t{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    };
    auto read_x = [&](const half_t* C, int tb) __attribute__((always_inline)) { return *reinterpret_cast<const half8_t*>(C + xoff[tb]); };

    float16_t acc[NTB][2];      // [token block][column block]
    float ss[NTB];
#pragma unroll
    for (int tb = 0; tb < NTB; ++tb) {
        ss[tb] = 0.f;
#pragma unroll
        for (int nb = 0; nb < 2; ++nb)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[tb][nb][r] = 0.f;
    }
    const bool stats = NORM > 0 && tn == 0;

    // Step s: stage s's operands are in wa / xb; those of stage s+1 (slot Cn) are read into wn / xn behind the MFMAs, and
    // stage s's own slot F is refilled with stage s+4.  Stage s+1 has landed: behind its requests only those of stages
    // s+2 and s+3 have been issued.  lgkmcnt(0): this wave's reads of stage s have returned, so no refill overtakes them.
    auto step = [&](int s, half8_t (&wa)[2], half8_t (&xb)[NTB], half8_t (&wn)[2], half8_t (&xn)[NTB], const half_t* Cn,
                    half_t* F, half8_t& g) __attribute__((always_inline)) {
        constexpr int kBehind = 2 * NL;
        __builtin_amdgcn_s_waitcnt(0x0070 | (kBehind & 15) | ((kBehind >> 4) << 14));
        __builtin_amdgcn_s_barrier();        // (a bare barrier: the loads in flight must stay in flight)
        __builtin_amdgcn_sched_barrier(0);
        half8_t xg[NTB];                     // (gamma is used up before its slot of the ring is refilled)
#pragma unroll
        for (int tb = 0; tb < NTB; ++tb) { if constexpr (NORM == 2) xg[tb] = xb[tb] * g; else xg[tb] = xb[tb]; }
        // With eight MFMAs a stage its requests go out one by one behind them: all at once they keep the wave from issuing
        // anything else (4096 -> 6144, us at once / dealt out, with norm and gamma; without: 300 tokens 45.4 / 41.3; 30.4 / 29.1, 512
        // 46.0 / 43.3; 39.8 / 38.6, 640 51.3 / 49.2; 40.2 / 39.0; the tiles of two and four MFMAs: the same).
        constexpr bool kDeal = NTB == 4;
        if constexpr (!kDeal) fetch(s + 4, F, g);
        auto deal = [&](int mfma) __attribute__((always_inline)) {
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int n = 0; n < NL; ++n) if (kDeal && n * 2 * NTB / NL == mfma) request(n, s + 4, F, g);
            __builtin_amdgcn_sched_barrier(0);
        };
#pragma unroll
        for (int tb = 0; tb < NTB; ++tb) {
            acc[tb][0] = mfma32(wa[0], xg[tb], acc[tb][0]);
            if (tb == 0) { wn[0] = read_w(Cn, 0); if (NTB == 1) wn[1] = read_w(Cn, 1); }
            if (tb == 1) wn[1] = read_w(Cn, 1);
            if (NTB <= 2) xn[tb] = read_x(Cn, tb);
            else if (tb >= 2) { xn[2 * tb - 4] = read_x(Cn, 2 * tb - 4); xn[2 * tb - 3] = read_x(Cn, 2 * tb - 3); }
            deal(2 * tb);
            acc[tb][1] = mfma32(wa[1], xg[tb], acc[tb][1]);
            if (stats) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const half2_t p = {xb[tb][2 * e], xb[tb][2 * e + 1]};
                    ss[tb] = __builtin_amdgcn_fdot2(p, p, ss[tb], false);
                }
            }
            deal(2 * tb + 1);
        }
    };
    half8_t waA[2], xbA[NTB], waB[2], xbB[NTB];
    fetch(0, S0, g0); fetch(1, S1, g1); fetch(2, S2, g2); fetch(3, S3, g3);
    {
        constexpr int kBehind = 3 * NL;
        __builtin_amdgcn_s_waitcnt(0x0f70 | (kBehind & 15) | ((kBehind >> 4) << 14));
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) waA[nb] = read_w(S0, nb);
#pragma unroll
        for (int tb = 0; tb < NTB; ++tb) xbA[tb] = read_x(S0, tb);
    }
    for (int s = 0; s < nst; s += 4) {       // whole turns of the ring: stages past hidden are zeros and add nothing
        step(s, waA, xbA, waB, xbB, S1, S0, g0);
        step(s + 1, waB, xbB, waA, xbA, S2, S1, g1);
        step(s + 2, waA, xbA, waB, xbB, S3, S2, g2);
        step(s + 3, waB, xbB, waA, xbA, S0, S3, g3);
    }
    __builtin_amdgcn_s_waitcnt(0x0070);      // the refills past the end have landed, the last reads have returned
    __syncthreads();
    if (stats) {
#pragma unroll
        for (int tb = 0; tb < NTB; ++tb) {
            const float s = half_sum(ss[tb]);
            if (h == 0) ss_part[kq][(tm * NTB + tb) * 32 + c] = s;
        }
    }

    // ---- add the partial tiles of the four contraction steps, one 32 x 32 block per wave at a time: float [32 tokens]
    // [32 columns], the 4-float chunks of a row XOR-swizzled by the token; then 16 bytes of output per thread
    constexpr int PPS = (MT + NT) * SK * 2 / 4096;      // 4 KB pieces per stage array
    static_assert(2 * PPS >= NW, "the partial blocks take two stage arrays at most");
    auto piece = [&](int p) __attribute__((always_inline)) {
        return reinterpret_cast<float*>(p < PPS ? S0 : S1) + (p < PPS ? p : p - PPS) * 1024;
    };
#pragma unroll
    for (int tb = 0; tb < NTB; ++tb) {
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) {
            float* mine = piece(wave);
#pragma unroll
            for (int r4 = 0; r4 < 4; ++r4)
                *reinterpret_cast<float4_t*>(&mine[c * 32 + (((2 * r4 + h) ^ (c & 7)) << 2)]) =
                    float4_t{acc[tb][nb][4 * r4], acc[tb][nb][4 * r4 + 1], acc[tb][nb][4 * r4 + 2], acc[tb][nb][4 * r4 + 3]};
            __syncthreads();
            if (tid < TM * TN * 128) {
                const int oc = tid & 3, tr = (tid >> 2) & 31, wn = (tid >> 7) % TN, wm = (tid >> 7) / TN;
                const int trow = (wm * NTB + tb) * 32 + tr, t = m0 + trow;
                float4_t u = {0.f, 0.f, 0.f, 0.f}, v = {0.f, 0.f, 0.f, 0.f};
                float sq = 0.f;
#pragma unroll
                for (int k = 0; k < KQ; ++k) {
                    const float* b = piece((wm * TN + wn) * KQ + k);
                    u += *reinterpret_cast<const float4_t*>(&b[tr * 32 + (((2 * oc) ^ (tr & 7)) << 2)]);
                    v += *reinterpret_cast<const float4_t*>(&b[tr * 32 + (((2 * oc + 1) ^ (tr & 7)) << 2)]);
                    if constexpr (NORM > 0) sq += ss_part[k][trow];
                }
                const float rstd = NORM > 0 ? 1.0f / __builtin_sqrtf(sq / (float)a.K + a.eps) : 1.0f;
                const int n = n0 + wn * 64 + nb * 32 + 8 * oc;
                if (t < a.T && n < P.n) {
                    const int64_t o_off = (int64_t)(n / a.head_dim) * P.stride_h + (int64_t)t * P.stride_s + (n % a.head_dim);
                    half8_t ov;
#pragma unroll
                    for (int e = 0; e < 4; ++e) { ov[e] = (half_t)(u[e] * rstd); ov[4 + e] = (half_t)(v[e] * rstd); }
                    if (P.addend) {
                        const half8_t ad = *reinterpret_cast<const half8_t*>(P.addend + o_off);
#pragma unroll
                        for (int e = 0; e < 8; ++e) ov[e] = (half_t)((float)ov[e] + (float)ad[e]);
                    }
                    *reinterpret_cast<half8_t*>(P.out + o_off) = ov;
                }
            }
            __syncthreads();
        }
    }
#endif
}

int64_t prenorm_qkv_mid_tiles(const GemmArgs& a, int mt, int nt) {
    int64_t panels = 0;
    for (int i = 0; i < 3; ++i) panels += (a.p[i].n + nt - 1) / nt;
    return ((int64_t)a.T + mt - 1) / mt * panels;
}

template <int NTB, int TM, int TN, bool STREAM>
static int launch_mid(GemmArgs a, hipStream_t stream) {
    constexpr int MT = TM * NTB * 32, NT = TN * 64;
    a.n_mtiles = (a.T + MT - 1) / MT;
    int t0 = 0;
    for (int i = 0; i < 3; ++i) { a.p[i].tile0 = t0; t0 += (a.p[i].n + NT - 1) / NT; }
    a.n_panels = t0;
    const int64_t grid = (int64_t)8 * ((t0 + 7) / 8) * a.n_mtiles;
    if (grid > 0x7fffffffLL) return TRN_E_SHAPE;
    auto* kernel = !a.norm ? prenorm_qkv_mid_kernel<NTB, TM, TN, 0, STREAM> : !a.gamma ? prenorm_qkv_mid_kernel<NTB, TM, TN, 1, STREAM>
                                                                                   : prenorm_qkv_mid_kernel<NTB, TM, TN, 2, STREAM>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(512), 0, stream, a);
    return hipGetLastError() == hipSuccess ? TRN_OK : TRN_E_LAUNCH;
}

int launch_prenorm_qkv_mid(const GemmArgs& a, int mt, int nt, hipStream_t stream) {
    if (nt == 128) return launch_mid<4, 1, 2, false>(a, stream);
    if (a.T <= mt && weights_stream(a)) return mt == 128 ? launch_mid<2, 2, 1, true>(a, stream) : launch_mid<1, 2, 1, true>(a, stream);
    return mt == 128 ? launch_mid<2, 2, 1, false>(a, stream) : launch_mid<1, 2, 1, false>(a, stream);
}

}  // namespace trn
