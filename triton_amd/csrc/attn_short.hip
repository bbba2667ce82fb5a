// Attention with key statistics (KeyFormer key scores, RoCo sums) on short prompts: 33 to 128 queries, at most 128 keys.
//
// Two launches of some 6 us each -- the forward, then statistics that need its row normalisers -- are nothing but latencies
// at these sizes: a launch, the first loads, a chain of a few MFMAs and exponentials, the ends.  Here a workgroup owns a
// (batch, head): four waves of 32 queries, the whole of K and V in LDS from the start.  A row's scores stay in registers (four
// 32-key blocks, twice with noise), so the maximum and the normaliser are exact in one go, nothing is multiplied twice, and
// what the statistics need is there when the normalisers are: each wave adds its queries' probabilities up over the lanes
// (4 KB of its own LDS), and the four waves' sums meet in the K tile.
//
// Formulation and operand layouts are those of the decode kernel: S^T = K Q^T, P^T taken from the S^T accumulator, V^T through
// the transposing LDS read.  Noise comes in whole 128-byte row pieces per eight lanes and is turned into the accumulator
// layout through the wave's 4 KB (as in the statistics kernel).
//
// What bounds it: launch, loads and the longest wave's chain.  us, two launches / this, KeyFormer with fp16 noise; RoCo: 32 / 8
// heads of 128, 33 tokens 12.0 / 6.2; 11.3 / 6.1, 64 12.1 / 6.4; 11.1 / 6.1, 100 14.5 / 9.4; 12.8 / 8.8, 8 x 128 18.3 / 11.6; 15.3 /
// 10.4; 71 / 1 heads of 64, 100 tokens 16.4 / 8.2; 11.8 / 7.7, 8 x 128 26.8 / 17.9; 19.6 / 12.2; 16 heads of 64, 128 tokens 12.6 /
// 8.1; 10.7 / 7.6.
#include <type_traits>
#include "attn.h"

namespace trn {

constexpr int kShort = 128;       // queries and keys at most

// NZ: 0 no noise, 1 fp32 noise, 2 fp16 noise
template <int D, int NZ>
__global__ __launch_bounds__(256, 2) void attn_short_kernel(const AttnArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)   // buffer descriptors and LDS-load builtins exist in the device pass only
    constexpr bool NOISE = NZ != 0, N16 = NZ == 2;
    constexpr int NS = D / 16, NDB = D / 32, CPR = D / 8, RPI = 64 / CPR, NB = kShort / 32, NI = kShort / (4 * RPI);
    __shared__ __attribute__((aligned(1024))) half_t Ks[kShort * D];
    __shared__ __attribute__((aligned(1024))) half_t Vs[kShort * D];
    __shared__ __attribute__((aligned(1024))) float Area[4 * 1024];

    const int tid = threadIdx.x, lane = tid & 63, c = lane & 31, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int G = a.Hq / a.Hkv, nkv = a.B * a.Hkv;
    const int kvslot = blockIdx.x % nkv, g = blockIdx.x / nkv;
    const int b = kvslot / a.Hkv, kvh = kvslot % a.Hkv, head = kvh * G + g;
    const int off = a.Skv - a.Sq, q0 = 32 * wave, qrow = q0 + c;
    const int64_t bh = (int64_t)b * a.Hq + head;
    // this wave's key blocks: none without queries, and under a causal mask none past its last query's last key
    const int seen = a.causal ? min(a.Skv, min(q0 + 31, a.Sq - 1) + off + 1) : a.Skv;
    const int nb = q0 < a.Sq ? (seen + 31) / 32 : 0;

    // ---- everything is requested at once: Q (B operands), noise, and the waves' shares of K and V (rows past the end: zeros)
    half8_t qB[NS];
    {
        const half_t* qp = a.q + b * a.qb + head * a.qh + (int64_t)min(qrow, a.Sq - 1) * a.qs + 8 * h;
#pragma unroll
        for (int ks = 0; ks < NS; ++ks) qB[ks] = *reinterpret_cast<const half8_t*>(qp + ks * 16);
    }
    const int st_row = wave * RPI + lane / CPR, st_chunk = ((lane % CPR) ^ swz<D>(st_row)) * 16;
    const __amdgpu_buffer_rsrc_t krs = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(a.k + b * a.kb + kvh * a.kh), 0, (int)(((int64_t)(a.Skv - 1) * a.ks + D) * 2), 0x00020000);
    const __amdgpu_buffer_rsrc_t vrs = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(a.v + b * a.vb + kvh * a.vh), 0, (int)(((int64_t)(a.Skv - 1) * a.vs + D) * 2), 0x00020000);
    fetch_tile<NI, D, 4>(krs, &Ks[wave * RPI * D], (int)(st_row * a.ks * 2) + st_chunk, 0, (int)(RPI * a.ks * 2));
    typedef typename std::conditional<N16, uint3_t, float4_t>::type noise_t;
    constexpr int nsz = N16 ? 2 : 4;
    const void* nbase = NOISE ? reinterpret_cast<const char*>(a.noise) + (b * a.nb + head * a.nh) * nsz : nullptr;
    const HalfNoise hn(nbase, N16 ? a.Sq : 1, N16 ? a.ns : 0, N16 ? a.Skv : 0);
    const __amdgpu_buffer_rsrc_t nrs = N16 ? hn.rs : __builtin_amdgcn_make_buffer_rsrc(
        (void*)nbase, 0, NOISE ? (int)(((int64_t)(a.Sq - 1) * a.ns + a.Skv) * 4) : 0, 0x00020000);
    noise_t gn[NOISE ? NB : 1][4];
    int nsh = 0;
    if constexpr (NOISE) {
        // load i of a block covers its query rows 8i .. 8i+7: lane -> row 8i + lane/8, keys 4*(lane%8) .. +3
        const int64_t first = (int64_t)(q0 + (lane >> 3)) * a.ns + 4 * (lane & 7);
        const int nvo = N16 ? hn.row(first, nsh) : (int)(first * 4), row8 = (int)(8 * a.ns * nsz);
#pragma unroll
        for (int kb = 0; kb < NB; ++kb)
            if (kb < nb) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if constexpr (N16) gn[kb][i] = __builtin_bit_cast(noise_t, __builtin_amdgcn_raw_buffer_load_b96(nrs, nvo, i * row8 + kb * 32 * nsz, 0));
                    else gn[kb][i] = __builtin_bit_cast(noise_t, __builtin_amdgcn_raw_buffer_load_b128(nrs, nvo, i * row8 + kb * 32 * nsz, 0));
                }
            }
    }
    fetch_tile<NI, D, 4>(vrs, &Vs[wave * RPI * D], (int)(st_row * a.vs * 2) + st_chunk, 0, (int)(RPI * a.vs * 2));
    __builtin_amdgcn_s_waitcnt(0x0f70);       // vmcnt(0)
    __syncthreads();

    // ---- scores, masked to -inf; with noise the perturbed ones too (these in the log2 domain)
    float* const area = Area + wave * 1024;
    float16_t s[NB], z[NOISE ? NB : 1];
    float m = -INFINITY, m2 = -INFINITY;
#pragma unroll
    for (int kb = 0; kb < NB; ++kb) {
        if (kb >= nb) continue;
#pragma unroll
        for (int r = 0; r < 16; ++r) s[kb][r] = 0.f;
#pragma unroll
        for (int ks = 0; ks < NS; ++ks)
            s[kb] = mfma32(*reinterpret_cast<const half8_t*>(&Ks[(kb * 32 + c) * D + (((2 * ks + h) ^ swz<D>(c)) << 3)]), qB[ks], s[kb]);
        // last key this lane's query sees, as an offset from the lane's first key of the block
        const int last = (a.causal ? min(qrow + off, a.Skv - 1) : a.Skv - 1) - (kb * 32 + 4 * h);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            s[kb][r] = 8 * (r / 4) + (r % 4) <= last ? s[kb][r] : -INFINITY;
            m = fmaxf(m, s[kb][r]);
        }
        if constexpr (NOISE) {
            // (LDS operations of one wave execute in order: no barrier between the two)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int r = 8 * i + (lane >> 3);
                float4_t v;
                if constexpr (N16) {
                    const half4_t hv = half_noise4(gn[kb][i], nsh);
                    v = float4_t{(float)hv[0], (float)hv[1], (float)hv[2], (float)hv[3]};
                } else v = gn[kb][i];
                *reinterpret_cast<float4_t*>(&area[(r * 8 + ((lane & 7) ^ ((r >> 1) & 7))) * 4]) = v;
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float4_t gq = *reinterpret_cast<const float4_t*>(&area[(c * 8 + ((2 * i + h) ^ ((c >> 1) & 7))) * 4]);
#pragma unroll
                for (int e = 0; e < 4; ++e) {           // a select: what lies past a row's last key may be anything, NaN included
                    z[kb][4 * i + e] = 8 * i + e <= last ? __builtin_fmaf(gq[e], a.c3, s[kb][4 * i + e] * a.c2) : -INFINITY;
                    m2 = fmaxf(m2, z[kb][4 * i + e]);
                }
            }
        }
    }
    m = half_max(m) * a.c1; m2 = half_max(m2);
    const float mref = m == -INFINITY ? 0.f : m, mref2 = m2 == -INFINITY ? 0.f : m2;      // (scores of minus infinity alone)

    // ---- probabilities, O^T = V^T P^T, the row's normaliser from exactly the values that multiply V
    float16_t oacc[NDB];
#pragma unroll
    for (int i = 0; i < NDB; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[i][r] = 0.f;
    float l = 0.f, l2 = 0.f;
    const half2_t ones = {(half_t)1.f, (half_t)1.f};
    const int rl = 4 * h + ((lane & 15) >> 2), rh = rl + 8, lc = 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1), sub = (lane & 1) * 4;
#pragma unroll
    for (int kb = 0; kb < NB; ++kb) {
        if (kb >= nb) continue;
        half8_t pB[2];
#pragma unroll
        for (int r = 0; r < 16; r += 2) {
            const half2_t pp = {(half_t)fast_exp2(__builtin_fmaf(s[kb][r], a.c1, -mref)), (half_t)fast_exp2(__builtin_fmaf(s[kb][r + 1], a.c1, -mref))};
            l = __builtin_amdgcn_fdot2(pp, ones, l, false);
            pB[r / 8][r % 8] = pp[0]; pB[r / 8][r % 8 + 1] = pp[1];
            if constexpr (NOISE) l2 += fast_exp2(z[kb][r] - mref2) + fast_exp2(z[kb][r + 1] - mref2);
        }
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int db = 0; db < NDB; ++db) {
                const half_t* vp = Vs + (kb * 32 + 16 * i) * D;
                const half4_t lo = lds_read_tr16(&vp[rl * D + (((db * 4 + lc) ^ swz<D>(rl)) << 3) + sub]);
                const half4_t hi = lds_read_tr16(&vp[rh * D + (((db * 4 + lc) ^ swz<D>(rh)) << 3) + sub]);
                oacc[db] = mfma32(half8_t{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]}, pB[i], oacc[db]);
            }
    }
    l = half_sum(l); l2 = half_sum(l2);
    if (qrow < a.Sq) {
        const float inv = 1.0f / l;
        half_t* orow = a.o + b * a.ob + head * a.oh + (int64_t)qrow * a.os + 4 * h;
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
            for (int r4 = 0; r4 < 4; ++r4)
                *reinterpret_cast<half4_t*>(orow + db * 32 + 8 * r4) = half4_t{
                    (half_t)(oacc[db][4 * r4] * inv), (half_t)(oacc[db][4 * r4 + 1] * inv), (half_t)(oacc[db][4 * r4 + 2] * inv), (half_t)(oacc[db][4 * r4 + 3] * inv)};
        if (h == 0) {
            if (a.lse) a.lse[bh * a.Sq + qrow] = (m + fast_log2(l)) * kLn2;
            if constexpr (NOISE) a.lse_pert[bh * a.Sq + qrow] = (m2 + fast_log2(l2)) * kLn2;
        }
    }

    // ---- statistics: this wave's sums over its queries, then over the waves (in the K tile, which everybody has left)
    const float lq = qrow >= a.Sq ? INFINITY : NOISE ? m2 + fast_log2(l2) : m + fast_log2(l);     // (lanes without a query add nothing)
    float* const sums = reinterpret_cast<float*>(Ks);              // [x, y][wave][key]
    __syncthreads();
#pragma unroll
    for (int kb = 0; kb < NB; ++kb) {
        float x = 0.f, y = 0.f;
        if (kb < nb) {
            float p[16];
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float t = NOISE ? z[NOISE ? kb : 0][r] : s[kb][r];
                p[r] = t == -INFINITY ? 0.f : fast_exp2(NOISE ? t - lq : __builtin_fmaf(t, a.c1, -lq));
            }
            put_sums(p, area, area + 512, lane);
            x = key_sum(area, area + 512, lane);
            if (a.col_sumsq) {
#pragma unroll
                for (int r = 0; r < 16; ++r) p[r] *= p[r];
                put_sums(p, area, area + 512, lane);
                y = key_sum(area, area + 512, lane);
            }
        }
        if ((lane & 1) == 0) {
            sums[wave * kShort + kb * 32 + key_of_sum(lane)] = x;
            sums[(4 + wave) * kShort + kb * 32 + key_of_sum(lane)] = y;
        }
    }
    __syncthreads();
    if (tid < a.Skv) {
        const float* p = sums + tid;
        float x = (p[0] + p[kShort]) + (p[2 * kShort] + p[3 * kShort]), y = (p[4 * kShort] + p[5 * kShort]) + (p[6 * kShort] + p[7 * kShort]);
        if (a.mean_std) mean_std_of(x, y, (float)(a.causal ? a.Sq - max(0, tid - off) : a.Sq));
        store_stat(a.col_sum, a.s16, bh * a.Skv + tid, x);
        store_stat(a.col_sumsq, a.s16, bh * a.Skv + tid, y);
    }
#endif
}

// (every form of these sizes gains, one head or hundreds, see above)
bool attn_short_suits(int seq_q, int seq_kv) { return seq_q > 32 && seq_q <= kShort && seq_kv <= kShort; }

hipError_t launch_attn_short(const AttnArgs& a, int head_dim, hipStream_t s) {
    const int64_t grid = (int64_t)a.B * a.Hq;
    if (grid > 0x7fffffffLL) return hipErrorInvalidValue;
    const dim3 g((unsigned)grid), t(256);
#define TRN_SHORT(D_) do { if (!a.noise) hipLaunchKernelGGL((attn_short_kernel<D_, 0>), g, t, 0, s, a); \
        else if (a.n16) hipLaunchKernelGGL((attn_short_kernel<D_, 2>), g, t, 0, s, a); else hipLaunchKernelGGL((attn_short_kernel<D_, 1>), g, t, 0, s, a); } while (0)
    if (head_dim == 128) TRN_SHORT(128); else TRN_SHORT(64);
#undef TRN_SHORT
    return hipGetLastError();
}

}  // namespace trn
