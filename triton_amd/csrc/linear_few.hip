// LoRA and the gated MLP of few tokens on little weight in one launch:
//
//     O = X W + (X A) B        O = gate(X W1) * (X W2)
//
// Two launches -- {O, D} = X {W, A} and O += D B; both products and their gate -- are two chains of memory latencies of 3 to 4 us
// each, however small, and the second waits for the first.  Here a workgroup owns 32 columns of O and forms what they need besides: all
// of D = X A, which its neighbours form as well (A and X come from L2), or the same columns of the second product.
//
// What bounds it: the latency of the first loads and, from some 100 KB a workgroup on, what a CU takes in.  Eight waves take the
// contraction in turns of 32 rows, as in prenorm_qkv_skinny.hip, but with up to four turns' loads on their way at once: so little
// weight has no order of DRAM pages to lose.  The last four turns have no loads behind them, so that 1024 rows pass without a loop.
// 16x16x32 MFMAs: at most 16 tokens fill half of a 32x32 one, and the sums of eight waves that pass through LDS are half as many (16
// tokens, 1024 x 512, rank 64 in 32x32x16 7.0 us, in 16x16x32 6.3, without the loads behind the last turns 5.9).
#include "prenorm_qkv.h"

namespace trn {

struct FewArgs {
    const half_t* x; const half_t* w; const half_t* a; const half_t* b; half_t* o;
    int T, K, n, r, n_panels, silu;
    int64_t ldx, ldw, lda, ldb, ldo;
};

// NR: blocks of 32 columns of the second matrix (A, or the panel of W2); TB: blocks of 16 tokens; PD: turns on their way
template <int NR, int TB, int PD, bool GATE>
__global__ __launch_bounds__(512, 2) void linear_few_kernel(const FewArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
    constexpr int NW = 8, NB = 1 + NR;                                 // waves, column blocks
    constexpr int CPR = 4 * NR, RPL = 64 / CPR, AL = 32 / RPL;         // second matrix: chunks per row, rows per load, loads
    constexpr int STAGE = NB * 1024 + TB * 512, DP = NR * 32 + 8;      // halfs of a wave's k-tile; pitch of D
    constexpr int SSZ = NW * STAGE * 2, RSZ = NW * NB * 8 * 64 * 4;
    __shared__ __attribute__((aligned(1024))) char smem[SSZ > RSZ ? SSZ : RSZ];
    __shared__ __attribute__((aligned(256))) half_t Dm[GATE ? 8 : TB * 16 * DP];
    __shared__ __attribute__((aligned(256))) half_t Bs[GATE ? 8 : NR * 32 * 32];

    const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // (the two panels of a 128-byte line go to one XCD, whose L2 then has the line for both)
    const int id = blockIdx.x, panel = 16 * (id >> 4) + 2 * (id & 7) + ((id >> 3) & 1);
    if (panel >= a.n_panels) return;
    const int n0 = 32 * panel, nkt = (a.K + 31) / 32;
    const int64_t t0 = (int64_t)blockIdx.y * (16 * TB);                // (the token tiles of a panel are on one XCD as well)
    const int T = min((int)(a.T - t0), 16 * TB);
    constexpr int kOut = 0x7ffffff0;                 // a byte offset past every buffer: the load returns zeros
    auto rows_of = [](const half_t* p, int64_t rows, int64_t pitch, int64_t cols) __attribute__((always_inline)) {
        return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, (int)(((rows - 1) * pitch + cols) * 2), 0x00020000);
    };
    const __amdgpu_buffer_rsrc_t xrs = rows_of(a.x + t0 * a.ldx, T, a.ldx, a.K), wrs = rows_of(a.w, a.K, a.ldw, a.n);
    const __amdgpu_buffer_rsrc_t ars = rows_of(a.a, a.K, a.lda, GATE ? a.n : a.r);
    const int wr = lane >> 2, wc = lane & 3, ar = lane / CPR, ac = lane % CPR;
    const int w_pitch = (int)a.ldw * 2, a_pitch = (int)a.lda * 2, acol = (GATE ? n0 : 0) + 8 * ac;
    const int w_vo = wr * w_pitch + (n0 + 8 * wc) * 2, a_vo = acol < (GATE ? a.n : a.r) ? ar * a_pitch + acol * 2 : kOut;
    int x_vo[TB];
#pragma unroll
    for (int i = 0; i < TB; ++i) x_vo[i] = 16 * i + wr < T ? (int)((16 * i + wr) * a.ldx * 2) + wc * 16 : kOut;

    // (unconditional, past the end as zeros: a load that may not be issued counts as absent when the compiler sizes its waits)
    half8_t wreg[PD][2], areg[PD][AL], xreg[PD][TB], breg;
    auto load = [](__amdgpu_buffer_rsrc_t rs, int vo, int so) __attribute__((always_inline)) {
        return __builtin_bit_cast(half8_t, __builtin_amdgcn_raw_buffer_load_b128(rs, vo, so, 0));
    };
    auto fetch = [&](int j, int kt) __attribute__((always_inline)) {
        const int k = 32 * min(kt, nkt), none = kt < nkt ? 0 : kOut;
        const bool drop = k + 8 * wc >= a.K;                   // (columns past hidden hold the next row's data)
#pragma unroll
        for (int i = 0; i < 2; ++i) wreg[j][i] = load(wrs, w_vo | none, (k + 16 * i) * w_pitch);
#pragma unroll
        for (int i = 0; i < AL; ++i) areg[j][i] = load(ars, a_vo | none, (k + RPL * i) * a_pitch);
#pragma unroll
        for (int i = 0; i < TB; ++i) xreg[j][i] = load(xrs, drop ? kOut : x_vo[i], k * 2);
    };

    // ---- this wave's part of LDS: the blocks of 32 rows of 64 bytes each, then X in rows of 64 bytes, chunk j at j ^ ((r/4) % 4)
    half_t* const Wm = reinterpret_cast<half_t*>(smem) + wave * STAGE;
    half_t* const Xm = Wm + NB * 1024;
    const int w_st = lane * 8, a_st = (1 + (ac >> 2)) * 1024 + ar * 32 + (ac & 3) * 8, x_st = wr * 32 + ((wc ^ ((wr >> 2) & 3)) << 3);
    const int x_ld = c * 32 + ((g ^ ((c >> 2) & 3)) << 3);
    // W^T through the transposing read: 16 columns, rows 8g + c/4 [+4]
    const int w_ld = (8 * g + (c >> 2)) * 32 + (c & 3) * 4;
    auto operand = [&](const half_t* block) __attribute__((always_inline)) {
        const half4_t lo = lds_read_tr16(block + w_ld), hi = lds_read_tr16(block + w_ld + 4 * 32);
        return half8_t{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    };
    auto mfma16 = [](half8_t x, half8_t y, float4_t z) __attribute__((always_inline)) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(x, y, z, 0, 0, 0); };

    const float4_t zero = {0.f, 0.f, 0.f, 0.f};
    float4_t acc[TB][2 * NB];
#pragma unroll
    for (int tb = 0; tb < TB; ++tb)
#pragma unroll
        for (int nb = 0; nb < 2 * NB; ++nb) acc[tb][nb] = zero;

    if constexpr (!GATE) {                           // this panel's columns of B: 16 rows a wave
        const __amdgpu_buffer_rsrc_t brs = rows_of(a.b, a.r, a.ldb, a.n);
        const int k = 16 * wave + wr;
        breg = load(brs, wave < 2 * NR && k < a.r ? (int)(k * a.ldb * 2) + (n0 + 8 * wc) * 2 : kOut, 0);
    }
#pragma unroll
    for (int j = 0; j < PD; ++j) {
        fetch(j, wave + NW * j);
        __builtin_amdgcn_sched_barrier(0);           // (in this order: the loop's first wait is for the first turn alone)
    }
    auto turn = [&](int j, int ahead) __attribute__((always_inline)) {       // ahead: the turn to ask for in its place, -1: none
#pragma unroll
        for (int i = 0; i < 2; ++i) *reinterpret_cast<half8_t*>(Wm + i * 512 + w_st) = wreg[j][i];
#pragma unroll
        for (int i = 0; i < AL; ++i) *reinterpret_cast<half8_t*>(Wm + i * RPL * 32 + a_st) = areg[j][i];
#pragma unroll
        for (int i = 0; i < TB; ++i) *reinterpret_cast<half8_t*>(Xm + i * 512 + x_st) = xreg[j][i];
        __builtin_amdgcn_sched_barrier(0);
        if (ahead >= 0) fetch(j, ahead);
        __builtin_amdgcn_sched_barrier(0);
        half8_t xv[TB];
#pragma unroll
        for (int tb = 0; tb < TB; ++tb) xv[tb] = *reinterpret_cast<const half8_t*>(Xm + tb * 512 + x_ld);
#pragma unroll
        for (int nb = 0; nb < 2 * NB; ++nb) {
            const half8_t wv = operand(Wm + (nb >> 1) * 1024 + (nb & 1) * 16);
#pragma unroll
            for (int tb = 0; tb < TB; ++tb) acc[tb][nb] = mfma16(wv, xv[tb], acc[tb][nb]);
        }
    };
    int kt = wave;
    for (; kt + NW * PD < nkt; kt += NW * PD)
#pragma unroll
        for (int j = 0; j < PD; ++j) turn(j, kt + NW * (j + PD));
#pragma unroll
    for (int j = 0; j < PD; ++j)
        if (kt + NW * j < nkt) turn(j, -1);
    if constexpr (!GATE)
        if (wave < 2 * NR) *reinterpret_cast<half8_t*>(Bs + wave * 512 + w_st) = breg;

    // ---- the eight waves' partial results: wave w finishes register w % 4 of the blocks' 16 columns number w / 4, which is column
    // col of them
    float* const red = reinterpret_cast<float*>(smem);
    const int col = 16 * (wave >> 2) + 4 * g + (wave & 3);
    float sum[TB][NB];
#pragma unroll
    for (int tb = 0; tb < TB; ++tb) {
        __syncthreads();
#pragma unroll
        for (int nb = 0; nb < 2 * NB; ++nb)
#pragma unroll
            for (int r = 0; r < 4; ++r) red[((wave * NB * 2 + nb) * 4 + r) * 64 + lane] = acc[tb][nb][r];
        __syncthreads();
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            float v = 0.f;
#pragma unroll
            for (int w = 0; w < NW; ++w) v += red[((w * NB + nb) * 8 + wave) * 64 + lane];
            sum[tb][nb] = v;
        }
    }
    // ---- every product is rounded to fp16, as a separate one would leave it
    if constexpr (!GATE) {
#pragma unroll
        for (int tb = 0; tb < TB; ++tb)
#pragma unroll
            for (int nb = 1; nb < NB; ++nb) {
                const int d = 32 * (nb - 1) + col;   // (columns past the rank: zeros also where X is no number)
                Dm[(16 * tb + c) * DP + d] = d < a.r ? (half_t)sum[tb][nb] : (half_t)0.f;
            }
        __syncthreads();
    }
#pragma unroll
    for (int tb = 0; tb < TB; ++tb) {
        half_t o;
        if constexpr (GATE) {
            const float u = (float)(half_t)sum[tb][0], sg = 1.0f / (1.0f + fast_exp2(-u * kLog2e));
            o = (half_t)((a.silu ? u * sg : sg) * (float)(half_t)sum[tb][1]);
        } else {
            float4_t p = zero;
#pragma unroll
            for (int ks = 0; ks < NR; ++ks)
                p = mfma16(operand(Bs + ks * 1024 + 16 * (wave >> 2)), *reinterpret_cast<const half8_t*>(Dm + (16 * tb + c) * DP + 32 * ks + 8 * g), p);
            const float q = wave & 2 ? (wave & 1 ? p[3] : p[2]) : (wave & 1 ? p[1] : p[0]);
            o = (half_t)((float)(half_t)q + (float)(half_t)sum[tb][0]);
        }
        const int t = 16 * tb + c;
        if (t < T && n0 + col < a.n) a.o[(t0 + t) * a.ldo + n0 + col] = o;
    }
#endif
}

// Where that is faster than two launches: up to what depth, by what a workgroup takes in beside its own panel (all of A; the second
// panel, of which there are half as many workgroups as the two launches have).  Up to 4096 columns; us in a graph, weights from beyond the
// L2s, tokens: depth x columns two launches / one (called one by one, the two take up to 2 us more of the host's time):
//   LoRA, rank 33 to 64   12: 968 x 512 5.8 / 5.6, 1112 x 3712 8.1 / 7.3, 4: 1320 x 1920 8.4 / 7.8; but 12: 1096 x 384 5.8 / 6.6, 16: 1176 x 64 5.4 / 6.2
//                         24: 600 x 768 6.0 / 5.9, 32: 1048 x 3864 10.1 / 9.6; but 24: 920 x 640 6.2 / 7.2, 1040 x 256 6.3 / 6.9
//   rank 8 to 32          16: 256 x 256 5.9 / 3.8, 2048 x 1024 7.8 / 6.4, 3248 x 1160 12.4 / 9.9; but 8: 3104 x 72 8.3 / 9.1, 12: 2640 x 256 7.2 / 9.1
//                         32: 1024 x 4096 7.6 / 5.8, 31: 2088 x 752 11.8 / 10.2; but 32: 1592 x 384 7.3 / 8.1, 17: 2240 x 128 6.9 / 9.0
//   rank 65 to 128        3: 696 x 3552 7.9 / 7.7; but 12: 648 x 128 5.3 / 6.1, 16: 4096 x 1024 9.8 / 20.7; 20: 256 x 3800 7.4 / 6.6; but 17: 328 x 128 5.2 / 6.0
//   gated MLP             4: 936 -> 1024 5.8 / 4.2, 1: 968 -> 3928 9.0 / 6.9, 9: 1336 -> 256 5.5 / 4.9; but 16: 1536 -> 4096 8.9 / 9.1
//                         28: 1088 -> 128 5.9 / 5.3, 25: 968 -> 4008 9.7 / 8.3; but 24: 952 -> 768 6.2 / 6.9
//                         rows that do not begin on whole lines, where few panels take in two lines a row: 4: 936 -> 240 5.2 / 4.5, 32: 720 -> 224 5.5 / 5.2;
//                         but 1: 1056 -> 184 5.4 / 6.0, 12: 1584 -> 176 6.7 / 8.1, 8: 1504 -> 120 5.5 / 7.6, 24: 1048 -> 168 5.7 / 7.2
// By columns up to 64, 128, 256, ... 4096; tokens up to 16, 32; rows of W at a pitch of whole lines, or not.
static int few_depth(int64_t tokens, int64_t n, int64_t ldw, int64_t rank, bool gate) {
    static constexpr short gated[2][7][2] = {{{1640, 1640}, {1640, 1080}, {1400, 800}, {1590, 1100}, {1340, 1260}, {1340, 1400}, {1280, 1280}},
                                             {{1040, 1040}, {1090, 1030}, {1040, 740}, {1090, 760}, {760, 860}, {1050, 1050}, {1024, 1024}}};
    static constexpr short r32[2][7][2] = {{{2480, 2480}, {2250, 2480}, {2250, 3584}, {2500, 3584}, {3584, 3584}, {3584, 3584}, {3584, 3584}},
                                           {{1550, 1550}, {1400, 1690}, {1400, 1800}, {1400, 1800}, {2360, 2360}, {2360, 2360}, {2360, 2560}}};
    static constexpr short r64[2][7][2] = {{{910, 910}, {1000, 1000}, {950, 950}, {1040, 1040}, {1070, 1300}, {1440, 1448}, {1448, 1448}},
                                           {{430, 430}, {640, 640}, {600, 760}, {640, 640}, {600, 700}, {640, 1080}, {1050, 1050}}};
    static constexpr short r128[2][7][2] = {{{420, 420}, {500, 500}, {500, 540}, {520, 520}, {480, 500}, {440, 600}, {560, 704}},
                                            {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 280}, {0, 320}, {0, 448}}};
    if (!gate && rank > 128) return 0;
    int wide = 0;
    while (wide < 6 && n > 64 << wide) ++wide;
    return (gate ? gated : rank <= 32 ? r32 : rank <= 64 ? r64 : r128)[tokens > 16][wide][ldw % 64 != 0];
}

// More than 32 tokens are tiles of 32, of which every CU has one at most (a panel's read its weights from the same L2): the two launches then
// take several us longer, and only all of A for a large rank makes up for it.  Ranks of up to 32 on little depth bear two a CU.
//   LoRA, rank 8 to 24   53 tokens, 328 x 272 8.0 / 4.9; 72, 1064 x 272 11.3 / 6.1; 145, 3816 x 328 25.4 / 15.0; 401, 576 x 432 10.6 / 5.6; 76, 688 x 2064 10.9 / 6.0; two a CU:
//                        71, 328 x 2848 10.2 / 7.6, 497, 568 x 816 11.1 / 9.5, 178, 968 x 1904 12.8 / 11.3; but 361, 1984 x 824 17.3 / 17.8, 449, 712 x 1240 (720 tiles) 12.1 / 14.1
//   rank 33 to 64        62 tokens, 512 x 1000 8.3 / 5.1; 177, 2984 x 448 16.1 / 14.4; 55, 1512 x 1256 11.1 / 10.6; 36, 4064 x 576 14.0 / 16.0; two a CU 317, 672 x 1056 10.8 / 12.4
//   rank 65 to 128       52 tokens, 304 x 784 8.5 / 6.7; 180, 472 x 504 10.4 / 7.5; 149, 656 x 1160 10.9 / 9.5; but 36, 824 x 512 8.6 / 9.1, 118, 2712 x 360 16.1 / 17.8
//   gated MLP            50 tokens, 424 -> 288 6.4 / 4.8; 88, 4000 -> 640 18.5 / 16.6; 47, 1352 -> 3024 12.9 / 10.2; 34, 4064 -> 728 17.8 / 18.6; 476, 384 -> 416 7.5 / 5.2; two a CU 365, 488 -> 608 7.7 / 8.8,
//                        82, 1264 -> 3248 13.2 / 16.7
//   few columns of up to 64 tokens, where the two launches do not take longer yet: LoRA, rank 64 54, 1296 x 128 8.4 / 9.4, 43, 1552 x 320 9.4 / 10.5; rank 128 50, 688 x 320
//                        7.9 / 8.5, 41, 552 x 1408 7.5 / 7.9; gated MLP 39, 1184 -> 144 7.1 / 8.1, 56, 1376 -> 80 7.4 / 8.5
static bool few_suits(int64_t tokens, int64_t hidden, int64_t n, int64_t ldw, int64_t rank, bool gate) {
    if (n > 4096) return false;
    if (tokens > 32) {
        const int64_t tiles = (n + 511) / 512 * 16 * ((tokens + 31) / 32);      // (as launch_few() has them)
        int64_t deep = 4096;
        if (tokens <= 64 && (gate || rank > 32)) deep = gate ? (n <= 256 ? 1000 : 3072) : n <= 384 ? 1100 : 3072;
        return hidden <= deep && (tiles <= 256 ? gate || rank <= 64 || (rank <= 128 && hidden <= (tokens <= 64 ? 540 : 704)) : !gate && rank <= 32 && hidden <= 1000 && tiles <= 512);
    }
    return hidden <= few_depth(tokens, n, ldw, rank, gate);
}

template <int NR, int PD, bool GATE>
static int launch_few(FewArgs a, hipStream_t stream) {
    a.n_panels = (a.n + 31) / 32;
    const dim3 g((unsigned)((a.n_panels + 15) / 16 * 16), (unsigned)((a.T + 31) / 32)), t(512);
    if (a.T <= 16) hipLaunchKernelGGL((linear_few_kernel<NR, 1, PD, GATE>), g, t, 0, stream, a);
    else hipLaunchKernelGGL((linear_few_kernel<NR, 2, PD, GATE>), g, t, 0, stream, a);
    return hipGetLastError() == hipSuccess ? TRN_OK : TRN_E_LAUNCH;
}

}  // namespace trn

extern "C" int trn_lora_f16(const void* x, int64_t tokens, int64_t hidden, int64_t ldx, const void* w, int64_t n, int64_t ldw,
                            const void* a, int64_t r, int64_t lda, const void* b, int64_t ldb, void* out, int64_t ldo,
                            void* d, int64_t ldd, void* stream) {
    using namespace trn;
    GemmArgs first, second;
    const void *w1[] = {w, a}, *w2[] = {b}, *ad[] = {out};
    void *o1[] = {out, d}, *o2[] = {out};
    const int64_t n1[] = {n, r}, l1[] = {ldw, lda}, p1[] = {ldo, ldd}, n2[] = {n}, l2[] = {ldb}, p2[] = {ldo};
    int st = linear_args(first, x, tokens, hidden, ldx, 2, w1, n1, l1, o1, p1, nullptr);
    if (st != TRN_OK) return st;
    st = linear_args(second, d, tokens, r, ldd, 1, w2, n2, l2, o2, p2, ad);
    if (st != TRN_OK || tokens == 0) return st;
    if (few_suits(tokens, hidden, n, ldw, r, false)) {
        const FewArgs f{(const half_t*)x, (const half_t*)w, (const half_t*)a, (const half_t*)b, (half_t*)out,
                        (int)tokens, (int)hidden, (int)n, (int)r, 0, 0, ldx, ldw, lda, ldb, ldo};
        hipStream_t s = (hipStream_t)stream;
        return r <= 32 ? launch_few<1, 4, false>(f, s) : r <= 64 ? launch_few<2, 4, false>(f, s) : launch_few<4, 2, false>(f, s);
    }
    st = launch_projections(first, (hipStream_t)stream);
    return st != TRN_OK ? st : launch_projections(second, (hipStream_t)stream);
}

extern "C" int trn_gated_mlp_f16(const void* x, int64_t tokens, int64_t hidden, int64_t ldx, const void* w1, int64_t ldw1,
                                 const void* w2, int64_t ldw2, int64_t n, void* out, int64_t ldo, void* c2, int64_t ldc,
                                 int32_t kind, void* stream) {
    using namespace trn;
    GemmArgs both;
    const void* w[] = {w1, w2};
    void* o[] = {out, c2};
    const int64_t ns[] = {n, n}, lw[] = {ldw1, ldw2}, lo[] = {ldo, ldc};
    if (kind != 0 && kind != 1) return TRN_E_SHAPE;
    int st = linear_args(both, x, tokens, hidden, ldx, 2, w, ns, lw, o, lo, nullptr);
    if (st != TRN_OK || tokens == 0) return st;
    if (few_suits(tokens, hidden, n, ldw1, 0, true)) {
        const FewArgs f{(const half_t*)x, (const half_t*)w1, (const half_t*)w2, nullptr, (half_t*)out,
                        (int)tokens, (int)hidden, (int)n, 0, 0, kind, ldx, ldw1, ldw2, 0, ldo};
        return launch_few<1, 4, true>(f, (hipStream_t)stream);
    }
    st = launch_projections(both, (hipStream_t)stream);
    return st != TRN_OK ? st : trn_gate_f16(out, c2, out, tokens, n, ldo, ldc, ldo, kind, stream);
}
