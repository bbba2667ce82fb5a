// Fused RMSNorm + Q/K/V projection for a handful of tokens (decode: at most 32; 64 on few weights), where the GEMM is a stream of the
// weight matrices through HBM and nothing else matters: 100 MB of W for 16 tokens at the Llama3-8B widths.
//
// Same arithmetic and MFMA mapping as the larger tilings (C^T = W^T X^T, 32x32x16 fp16 MFMAs, tokens padded to
// 32-wide blocks).  A workgroup owns a 64-column panel of one projection -- full 128-byte lines of every W row -- and
// its eight waves take the contraction in turns of SK rows: wave w's k-tiles are w, w + 8, ...  Nothing in the loop is
// shared between waves, so it has no barrier: a wave loads a k-tile of W and X into registers while it multiplies the
// one before, writes it to its private part of LDS when it arrives, and reads it back as MFMA operands (LDS operations
// of one wave execute in order).  The eight partial accumulators and sums of squares are added through LDS at the end.
//
// What bounds it is the order in which the rows reach HBM, not the bytes in flight.  A row of W lies in one DRAM page
// and its 64 panels belong to 64 workgroups: they profit from each other only while all of them walk the rows in
// lockstep.  Waves that own a quarter of the contraction each, as this kernel had them, or more than one k-tile in
// flight per wave pull the walk apart.  Reads alone, 100 MB cold, 128-byte panels of a 8192-byte pitch: 22.2 us with a
// quarter per wave, 20.5 in turns (16.7 at a pitch that is no power of two).  This kernel, us, quarters through LDS
// rings / now: 4096 -> 12288, 16 tokens 28.5 / 24.1, 32 tokens 31 / 25.5; 4544 -> 13632, 16 tokens 24.7 / 22.7;
// 1024 -> 3072 7.3 / 5.0; prefetching two or three k-tiles instead of one +0.5 and +1 us.
#include "prenorm_qkv.h"

namespace trn {

// XL: wave-wide loads that cover the tokens of a k-tile (rows of SK columns); NORM: 0 none, 1 without gamma, 2 with gamma
// SN: columns of a panel; NT: W is requested past the caches
template <int SK, int XL, int NORM, int SN, bool NT>
__global__ __launch_bounds__(512, 2) void prenorm_qkv_skinny_kernel(const GemmArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)   // buffer descriptors exist in the device pass only
    constexpr int NW = 8, NB = SN / 32, WC = SN / 8, WR = 64 / WC, WL = SK / WR;      // waves, column blocks; W: chunks per row, rows per load, loads
    constexpr int XC = SK / 8, XR = 64 / XC;                                           // X: chunks per row, rows per load
    constexpr int TB = (XL * XR + 31) / 32;                                            // blocks of 32 tokens
    static_assert((SK == 32 || SK == 64) && (SN == 32 || SN == 64) && TB <= 2, "k-tiles of 32 or 64 rows, at most 64 tokens");
    // [NW] W k-tiles, then [NW] X k-tiles (reads of token rows past the loaded ones stay inside: their results are never
    // stored); at the end the partial accumulators, 8 KB per wave
    constexpr int WSZ = NW * SK * SN, XSZ = NW * XL * XR * SK + (32 * TB - XL * XR) * SK, RSZ = NW * 16 * NB * 64 * 2;
    __shared__ __attribute__((aligned(1024))) half_t smem[WSZ + XSZ > RSZ ? WSZ + XSZ : RSZ];
    __shared__ __attribute__((aligned(256))) half_t Gs[NORM == 2 ? NW * SK : 8];
    __shared__ float ss_part[NW][32 * TB];

    const int tid = threadIdx.x, lane = tid & 63, c = lane & 31, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // (ids are dealt round-robin to the 8 XCDs: the two panels of a 128-byte line share an XCD's L2)
    const int id = blockIdx.x, panel = SN == 64 ? id : 16 * (id >> 4) + 2 * (id & 7) + ((id >> 3) & 1);
    if (SN == 32 && panel >= a.n_panels) return;
    const int pi = panel >= a.p[2].tile0 ? 2 : (panel >= a.p[1].tile0 ? 1 : 0);
    const ProjOut P = a.p[pi];
    const int n0 = (panel - P.tile0) * SN;
    if (SN == 32 && n0 >= P.n) return;               // (the place between an odd number of panels and the next matrix)
    const int nkt = (a.K + SK - 1) / SK;
    constexpr int kOut = 0x7ffffff0;                 // a byte offset past every buffer: the load returns zeros

    const __amdgpu_buffer_rsrc_t wrs = __builtin_amdgcn_make_buffer_rsrc(
        (void*)P.w, 0, (int)(((int64_t)(a.K - 1) * P.ldw + P.n) * 2), 0x00020000);
    const int wr = lane / WC, wc = lane % WC, xr = lane / XC, xc = lane % XC;
    const int w_vo = (int)(wr * P.ldw * 2) + (n0 + 8 * wc) * 2, w_step = (int)(WR * P.ldw * 2);
    const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc(
        (void*)a.x, 0, (int)(((int64_t)(a.T - 1) * a.ldx + a.K) * 2), 0x00020000);
    int x_vo[XL];
#pragma unroll
    for (int i = 0; i < XL; ++i) {
        const int t = XR * i + xr;
        x_vo[i] = t < a.T ? (int)(t * a.ldx * 2) + xc * 16 : kOut;
    }
    const __amdgpu_buffer_rsrc_t grs = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(NORM == 2 ? a.gamma : a.x), 0, NORM == 2 ? a.K * 2 : 0, 0x00020000);
    half8_t wreg[WL], xreg[XL], greg;
    auto fetch = [&](int s) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < WL; ++i) wreg[i] = __builtin_bit_cast(half8_t, __builtin_amdgcn_raw_buffer_load_b128(wrs, w_vo, (s * WL + i) * w_step, NT ? 2 : 0));
        // columns past hidden hold the next row's data: read zeros instead
        const bool drop = s * SK + 8 * xc >= a.K;
#pragma unroll
        for (int i = 0; i < XL; ++i) xreg[i] = __builtin_bit_cast(half8_t, __builtin_amdgcn_raw_buffer_load_b128(xrs, drop ? kOut : x_vo[i], s * SK * 2, 0));
        if constexpr (NORM == 2) greg = __builtin_bit_cast(half8_t, __builtin_amdgcn_raw_buffer_load_b128(grs, xc * 16, s * SK * 2, 0));
    };

    // ---- this wave's part of LDS.  W: chunk j of row r at j ^ swz<64>(r), a function of r % 16; as it is in rows of 64 bytes,
    // of which a transposing read takes four whole ones.  X: rows of 128 bytes:
    // chunk j at j ^ ((r/2) % 8), rows of 64 bytes: j ^ ((r/4) % 4).
    half_t* Wm = smem + wave * SK * SN;
    half_t* Xm = smem + WSZ + wave * XL * XR * SK;
    half_t* Gm = Gs + (NORM == 2 ? wave * SK : 0);
    auto xsw = [](int r) __attribute__((always_inline)) { return SK == 64 ? (r >> 1) & 7 : (r >> 2) & 3; };
    auto wsw = [](int r) __attribute__((always_inline)) { return SN == 64 ? swz<64>(r) : 0; };
    int w_st[2], x_st[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        w_st[i] = (WR * i + wr) * SN + ((wc ^ wsw(WR * i + wr)) << 3);
        x_st[i] = (XR * i + xr) * SK + ((xc ^ xsw(XR * i + xr)) << 3);          // (xsw repeats every 16 rows)
    }
    int woff_lo[NB], woff_hi[NB], xoff[SK / 16];     // W^T A-operand via the transposing read: rows 8h + (lane%16)/4 [+4] of a 16-row step
    {
        const int rl = 8 * h + ((lane & 15) >> 2), rh = rl + 4;
        const int lc = 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1), sub = (lane & 1) * 4;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            woff_lo[nb] = rl * SN + (((nb * 4 + lc) ^ wsw(rl)) << 3) + sub;
            woff_hi[nb] = rh * SN + (((nb * 4 + lc) ^ wsw(rh)) << 3) + sub;
        }
#pragma unroll
        for (int ks = 0; ks < SK / 16; ++ks) xoff[ks] = c * SK + (((2 * ks + h) ^ xsw(c)) << 3);
    }

    float16_t acc[TB][NB];
    float ss[TB];
#pragma unroll
    for (int tb = 0; tb < TB; ++tb) {
        ss[tb] = 0.f;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[tb][nb][r] = 0.f;
    }

    if (wave < nkt) fetch(wave);
    for (int kt = wave; kt < nkt; kt += NW) {
#pragma unroll
        for (int i = 0; i < WL; ++i) *reinterpret_cast<half8_t*>(&Wm[(i >> 1) * 2 * WR * SN + w_st[i & 1]]) = wreg[i];
#pragma unroll
        for (int i = 0; i < XL; ++i)
            *reinterpret_cast<half8_t*>(&Xm[SK == 64 ? (i >> 1) * 16 * SK + x_st[i & 1] : i * 16 * SK + x_st[0]]) = xreg[i];
        if (NORM == 2 && lane < XC) *reinterpret_cast<half8_t*>(&Gm[8 * lane]) = greg;
        __builtin_amdgcn_sched_barrier(0);
        if (kt + NW < nkt) fetch(kt + NW);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int ks = 0; ks < SK / 16; ++ks) {
            half8_t wa[NB];
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                const half4_t lo = lds_read_tr16(&Wm[ks * 16 * SN + woff_lo[nb]]);
                const half4_t hi = lds_read_tr16(&Wm[ks * 16 * SN + woff_hi[nb]]);
                wa[nb] = half8_t{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
            }
#pragma unroll
            for (int tb = 0; tb < TB; ++tb) {
                half8_t xv = *reinterpret_cast<const half8_t*>(&Xm[tb * 32 * SK + xoff[ks]]);
                if constexpr (NORM > 0) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const half2_t p = {xv[2 * e], xv[2 * e + 1]};
                        ss[tb] = __builtin_amdgcn_fdot2(p, p, ss[tb], false);
                    }
                    if constexpr (NORM == 2) xv = xv * *reinterpret_cast<const half8_t*>(&Gm[ks * 16 + 8 * h]);
                }
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) acc[tb][nb] = mfma32(wa[nb], xv, acc[tb][nb]);
            }
        }
    }

    // ---- add the eight waves' partial results through LDS
    float* red = reinterpret_cast<float*>(smem);             // [NW][16 NB registers][64 lanes], a block of 32 tokens at a time
    if constexpr (NORM > 0) {
#pragma unroll
        for (int tb = 0; tb < TB; ++tb) {
            const float s = half_sum(ss[tb]);                // both halves of a token's columns
            if (h == 0) ss_part[wave][32 * tb + c] = s;
        }
    }
    // wave w finishes accumulator registers FIN w .. FIN w + FIN-1: of column block w / (8 / NB), rows 8*(r/4) + 4h + r%4, token c
    constexpr int FIN = 2 * NB;
    typedef _Float16 fin_t __attribute__((ext_vector_type(FIN)));
    const int r0 = FIN * wave % 16, n = n0 + FIN * wave / 16 * 32 + 8 * (r0 / 4) + 4 * h + r0 % 4;
#pragma unroll
    for (int tb = 0; tb < TB; ++tb) {
        __syncthreads();
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int r = 0; r < 16; ++r) red[((wave * NB + nb) * 16 + r) * 64 + lane] = acc[tb][nb][r];
        __syncthreads();
        const int t = 32 * tb + c;
        float rstd = 1.0f;
        if constexpr (NORM > 0) {
            float sq = 0.f;
#pragma unroll
            for (int w = 0; w < NW; ++w) sq += ss_part[w][t];
            rstd = 1.0f / __builtin_sqrtf(sq / (float)a.K + a.eps);
        }
        if (t < a.T && n < P.n) {
            const int64_t o_off = (int64_t)(n / a.head_dim) * P.stride_h + (int64_t)t * P.stride_s + (n % a.head_dim);
            fin_t ad = {};
            if (P.addend) ad = *reinterpret_cast<const fin_t*>(P.addend + o_off);
            fin_t ov;
#pragma unroll
            for (int e = 0; e < FIN; ++e) {
                float v = 0.f;
#pragma unroll
                for (int w = 0; w < NW; ++w) v += red[(w * 16 * NB + FIN * wave + e) * 64 + lane];
                ov[e] = (half_t)((float)(half_t)(v * rstd) + (float)ad[e]);     // the product rounded to fp16 first, as a separate GEMM would leave it
            }
            *reinterpret_cast<fin_t*>(P.out + o_off) = ov;
        }
    }
#endif
}

// k-tiles of 32 rows up to 16 tokens (a shorter chain where hidden is small), of 64 beyond: 32 tokens x 64 bytes are half
// lines of X, and fetching those costs more than the shorter chain gains (4096 -> 12288, 32 tokens: 27.3 against 25.5 us).
template <int SN, bool NT>
static int launch_panels(GemmArgs a, hipStream_t stream) {
    int t0 = 0;
    for (int i = 0; i < 3; ++i) {
        // (a matrix begins with a whole pair, which one XCD has.  us, 16 tokens, weights cold, one behind the other / so: two matrices 4096 deep of
        // 4000 columns whose rows begin on whole lines 23.9 / 23.0, of 2080 17.5 / 17.15; rows at odd half lines and 1056 and fewer columns the same)
        if (SN == 32 && a.p[i].n > 0) t0 = (t0 + 1) & ~1;
        a.p[i].tile0 = t0;
        t0 += (a.p[i].n + SN - 1) / SN;
    }
    a.n_panels = t0;
    const dim3 g((unsigned)(SN == 64 ? t0 : (t0 + 15) / 16 * 16)), t(512);
    const int norm = !a.norm ? 0 : a.gamma ? 2 : 1;
#define TRN_SKINNY(SK_, XL_)                                                                                              \
    do {                                                                                                                  \
        if (norm == 0) hipLaunchKernelGGL((prenorm_qkv_skinny_kernel<SK_, XL_, 0, SN, NT>), g, t, 0, stream, a);              \
        else if (norm == 1) hipLaunchKernelGGL((prenorm_qkv_skinny_kernel<SK_, XL_, 1, SN, NT>), g, t, 0, stream, a);         \
        else hipLaunchKernelGGL((prenorm_qkv_skinny_kernel<SK_, XL_, 2, SN, NT>), g, t, 0, stream, a);                        \
    } while (0)
    if (a.T <= 16) TRN_SKINNY(32, 1);
    else if (a.T <= 24) TRN_SKINNY(64, 3);
    else if (SN == 64 || a.T <= 32) TRN_SKINNY(64, 4);
    else TRN_SKINNY(32, 4);
#undef TRN_SKINNY
    return hipGetLastError() == hipSuccess ? TRN_OK : TRN_E_LAUNCH;
}

// Panels of 32 columns while those of 64 would occupy at most half of the CUs: one CU takes in some 130 bytes a ns however many
// of its waves ask, so the time of few panels is their bytes per CU (X's among them).  The two panels of a 128-byte line go to
// one XCD, whose L2 then has the line for both; dealt out singly each line is fetched from HBM twice (4096 deep, 1056 columns,
// 16 tokens, with a second product of 32: 12.6 us in panels of 64, 15.5 of 32 dealt out singly, 9.5 so).  us, 64 / 32 columns, 16
// tokens, weights cold, launches in a graph: 1024 deep, 512 + 64 columns 5.5 / 4.8; 2048, 2080 + 2080 12.1 / 9.65; 4096, 4000 + 64 20.5 /
// 15.5, 4096 + 4096 25.2 / 22.9 (the last with 128 panels of 64); whole LoRA of 1024 x 512, rank 64, which is two launches, 9.3 / 8.4, and
// called one by one, where the host sets the pace as well, 10.1 / 8.2 to 9.7; but 4096, 12288 (192) 24.4 / 35.6, when the panels no longer
// run all at once.
int launch_prenorm_qkv_skinny(GemmArgs a, hipStream_t stream) {
    int panels = 0;
    for (int i = 0; i < 3; ++i) panels += (a.p[i].n + 63) / 64;
    if (a.T > 32) return launch_panels<32, false>(a, stream);
    return panels <= 128 ? launch_panels<32, false>(a, stream) : weights_stream(a) ? launch_panels<64, true>(a, stream) : launch_panels<64, false>(a, stream);
}

}  // namespace trn
