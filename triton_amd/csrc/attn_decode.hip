// Attention forward for at most 32 queries per head (decode-append: a few new tokens against a long cache), and for more
// of them where tiles of 32 queries are what it takes to occupy the chip (attn_decode_suits).
//
// With so few queries there is one 32-query MFMA block per head and the kernel is a stream of K and V through HBM.
// One workgroup per (batch, head, 32-query tile); its eight waves take the 32-key blocks round-robin, each with its own running
// max / normaliser / O^T accumulator, and the eight partial results are merged through LDS at the end (the usual
// log-sum-exp merge).  Formulation and register layouts are those of the prefill kernel: S^T = K Q^T with Q^T
// resident in registers, P^T taken from the S^T accumulator, V^T via the transposing LDS read.  K rows are what the
// A operand wants as they lie in memory, so K goes straight from global memory into registers (one block ahead);
// V goes global -> LDS into the wave's private two-stage ring.  Nothing in the loop is shared between waves, so the
// loop has no barrier; every load is issued unconditionally (blocks past the end read zeros, which are masked) so
// that the waits can be counted.
#include "attn.h"
#include "attn_decode_rules.h"
#include <mutex>
#include <type_traits>

typedef unsigned long long ulong2_t __attribute__((ext_vector_type(2)));

namespace trn {

constexpr int DNW = 8;    // waves per workgroup

// XOR swizzle of the 16-byte chunk index of a V row as wide as this workgroup's share of the head dimension
template <int DV> __device__ __forceinline__ int swzv(int r) {
    if constexpr (DV == 32) return (r >> 1) & 3;          // 4 chunks per 64-byte row
    else return swz<DV>(r);
}

// DS: the head dimension of V and O is shared out over DS workgroups per head (each computes all the scores, from
// all of K, but streams only its DV = D / DS columns of V and writes those columns of O).  One CU pulls 40 - 55 GB/s
// whatever its waves ask for, and with one workgroup per head that rate is what the kernel's time is made of; more
// workgroups per head without anything to hand over between them means fewer bytes through each CU.
// NZ: 0 no score perturbation, 1 fp32 noise, 2 fp16 noise, 3 none, and scores of normalised keys: a key's reciprocal root mean
// square multiplies its scores in fp32, and gamma_k is multiplied into the queries before they are rounded to fp16.  (Normalising
// the rows themselves costs ten times the vector instructions: us, a norm launch before / rows / scores: 16 heads of 64, 137 keys
// 9.2 / 7.0 / 6.8, 500 11.1 / 9.5 / 8.5; 32 heads of 128, 128 keys 11.3 / 9.5 / 9.2, 250 13.5 / 15.4 / 11.5.)
// 4, 5, 6: as 0, 1, 2 with key statistics on at most kept_blocks() key blocks per wave: the scores of a wave's blocks stay in its
// registers until the row normalisers are final, and the statistics need no second sweep over the keys and the noise.  With
// noise up to what the registers hold; without, the sums over the lanes cost what the sweep does from 1000 keys on.  Whole
// decode steps with 8 / 32 new tokens, us, sweep -> kept, 71 heads of 64 with fp16 noise: 200 keys 31.5 -> 30.2 / 35.3 -> 33.4,
// 1000 keys 37.1 -> 35.6 / 42.7 -> 40.0; 8 heads of 128: 15.1 -> 13.7 / 18.5 -> 16.0, 18.7 -> 17.4 / 22.2 -> 19.8; without noise
// 200 keys 14.2 -> 13.4 / 16.6 -> 14.9, but 71 heads and 1000 keys 34.7 -> 35.3 / 37.9 -> 38.4.
// 7: as 0, a workgroup one of n_split key shares, whose results the next launch merges.  (A form of its own: beside the unsplit one in
// the same kernel it cost that 0.1 of 4.3 us, 20 to 180 heads of 64, 30 tokens.)
constexpr int kept_blocks(int d, int ds, bool noise) { return !noise ? 2 : d == 128 && ds == 1 ? 3 : 6; }
template <int D, int DS, int NZ>
__global__ __launch_bounds__(DNW * 64, 1) void attn_decode_kernel(const AttnArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)   // buffer descriptors and LDS-load builtins exist in the device pass only
    constexpr bool SWEEP = NZ >= 8, PARTS = NZ == 7, KEEP = NZ >= 4 && !PARTS && !SWEEP, NOISE = NZ % 4 == 1 || NZ % 4 == 2, N16 = NZ % 4 == 2, KNORM = NZ == 3;
    constexpr int DV = D / DS;    // columns of V / O this workgroup owns
    constexpr int NS = D / 16;    // k-steps of S^T = K Q^T
    constexpr int NSV = DV / 16;  // (2 key halves) x (DV/32) MFMAs of P V
    constexpr int NDB = DV / 32;
    constexpr int CPR = DV / 8;   // 16-byte chunks per V row share
    constexpr int RPI = 64 / CPR; // rows per wave-wide 1 KB load
    constexpr int NI = 32 / RPI;  // such loads per 32-key V block
    // two V stages (each holds the eight waves' private parts), as two arrays: LDS reads are ordered after
    // outstanding global->LDS loads that may alias them, and only distinct variables are provably disjoint
    // (With the whole head dimension of V in one workgroup at head_dim 128 a V stage is 64 KB: one stage then, refilled
    // as soon as its block's P V is issued, so that the K area below still fits.)
    constexpr bool VSINGLE = D == 128 && DS == 1;
    __shared__ __attribute__((aligned(1024))) half_t Vs0[SWEEP ? 8 : DNW * 32 * DV];
    __shared__ __attribute__((aligned(1024))) half_t Vs1[SWEEP || VSINGLE ? 8 : DNW * 32 * DV];
    __shared__ float st_m[DNW][32], st_l[DNW][32], st_m2[DNW][32], st_l2[DNW][32];
    // K blocks are fetched as whole rows (a wave-wide load = 1 KB of consecutive bytes) and turned into MFMA operands
    // through a wave-private LDS area: a load whose lanes each take 16 bytes of their own row -- the operand layout --
    // is served at 16 bytes per clock (36 GB/s per CU measured), the row-wise one at 64 (130 GB/s).
    constexpr bool KLDS = true;
    constexpr int CPRK = D / 8;       // 16-byte chunks per K row
    constexpr int RPIK = 64 / CPRK;   // K rows per wave-wide load
    __shared__ __attribute__((aligned(1024))) half_t Kt[DNW * 32 * D];

    const int tid = threadIdx.x, lane = tid & 63, c = lane & 31, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // workgroup id -> (batch x head j, key share, column share).  The column shares of a head read the same K: their
    // ids are 8 apart, so that they sit on one XCD (ids are dealt to the 8 XCDs in turn) and share its L2.
    // So do the query tiles of a head, unless they are spread (decode_spread()); the last ones, with the most keys under a
    // causal mask, come first.
    // (the arguments of the start in one go: by itself the compiler asks for them where they are first needed, three memory latencies in a
    // row, of which divisions by the number of heads once hid one.  us, with the divisions / without / so: 8 heads of 64, 100 tokens 3.98 /
    // 4.23 / 3.90, 66, 30 tokens 4.20 / 4.45 / 4.16)
    asm volatile("" : : "s"(a.q), "s"(a.qb), "s"(a.q_norm), "s"(a.spread));
    int j, split = 0, dsl = 0, q0 = 0;
    const int BH = a.heads.all.d;
    if (a.n_qtiles > 1) {
        int qt;
        if (a.spread) {
            const int unit = (int)blockIdx.x / (8 * DS) * 8 + (int)blockIdx.x % 8;
            qt = a.heads.all.of(unit); j = unit - qt * BH; dsl = (int)blockIdx.x / 8 % DS;
        } else {
            const int per_grp = 8 * DS * a.n_qtiles, grp = (int)blockIdx.x / per_grp, rem = (int)blockIdx.x % per_grp;
            j = grp * 8 + rem % 8; qt = rem / (8 * DS); dsl = rem / 8 % DS;
        }
        if (j >= BH || qt >= a.n_qtiles) return;        // the last eight heads, or eight tiles, may be fewer
        q0 = 32 * (a.n_qtiles - 1 - qt);
    } else if constexpr (DS > 1) {
        const int grp = (int)blockIdx.x / (8 * DS), rem = (int)blockIdx.x % (8 * DS);
        j = grp * 8 + rem % 8; dsl = rem / 8;
        if (j >= BH) return;
    } else {
        j = blockIdx.x;
        if constexpr (PARTS || NOISE || SWEEP) { j = blockIdx.x / a.n_split; split = blockIdx.x % a.n_split; }
    }
    int b, kvh, g;
    a.heads.find(j, b, kvh, g);
    const int head = kvh * a.heads.G + g;
    const int off = a.Skv - a.Sq;                       // causal: query i sees keys <= i + off
    const int qrow = q0 + c;                            // this lane's query
    const int qrow_ld = qrow < a.Sq ? qrow : a.Sq - 1;

    // ---- Q^T B-operands: lane holds Q[qrow][ks*16 + 8h .. +7]; optional fused per-head RMSNorm of the row
    half8_t qB[NS];
    {
        const half_t* qp = a.q + b * a.qb + head * a.qh + (int64_t)qrow_ld * a.qs + 8 * h;
#pragma unroll
        for (int ks = 0; ks < NS; ++ks) qB[ks] = *reinterpret_cast<const half8_t*>(qp + ks * 16);
    }
    // (the norms' weights along with Q: one memory latency)
    half8_t gq[NS], gk[KNORM ? NS : 1];
    const bool use_gq = a.q_norm && a.gamma_q;
    if (use_gq) {
#pragma unroll
        for (int ks = 0; ks < NS; ++ks) gq[ks] = *reinterpret_cast<const half8_t*>(a.gamma_q + ks * 16 + 8 * h);
    }
    if constexpr (KNORM) {
#pragma unroll
        for (int ks = 0; ks < NS; ++ks) {
            if (a.gamma_k) gk[ks] = *reinterpret_cast<const half8_t*>(a.gamma_k + ks * 16 + 8 * h);
            else gk[ks] = half8_t{1, 1, 1, 1, 1, 1, 1, 1};
        }
    }
    // ---- K: block rows straight into registers as A operands (lane: key c of the block, columns ks*16 + 8h ..)
    const __amdgpu_buffer_rsrc_t krs = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(a.k + b * a.kb + kvh * a.kh), 0, (int)(((int64_t)(a.Skv - 1) * a.ks + D) * 2), 0x00020000);
    const int kvo = KLDS ? (int)((lane / CPRK) * a.ks * 2) + (lane % CPRK) * 16 : (int)(c * a.ks * 2) + 16 * h;
    const int kblk_bytes = (int)(32 * a.ks * 2), kpiece_bytes = (int)(RPIK * a.ks * 2);
    // With KLDS the registers hold piece i = rows i*RPIK .. +RPIK-1 of the block as they lie in memory (D/16 = NS
    // pieces); k_operands() below turns them into the operands in place.  Without it they are the operands.
    auto fetch_k = [&](int blk, half8_t (&ka)[NS]) __attribute__((always_inline)) {
#pragma unroll
        for (int ks = 0; ks < NS; ++ks) {
            if constexpr (KLDS)
                ka[ks] = __builtin_bit_cast(half8_t, __builtin_amdgcn_raw_buffer_load_b128(krs, kvo, blk * kblk_bytes + ks * kpiece_bytes, 0));
            else
                ka[ks] = __builtin_bit_cast(half8_t, __builtin_amdgcn_raw_buffer_load_b128(krs, kvo + ks * 32, blk * kblk_bytes, 0));
        }
    };
    // Rows into the wave's area (chunk j of row r at j ^ swz<D>(r): the write of a piece covers its 1 KB once, and
    // the 32 rows read back at one logical chunk touch every bank once), operands out of it.  LDS operations of one
    // wave execute in order and nobody else touches the area: no barrier.
    auto k_operands = [&](half8_t (&ka)[NS]) __attribute__((always_inline)) {
        if constexpr (KLDS) {
            half_t* kt = Kt + wave * 32 * D;
#pragma unroll
            for (int i = 0; i < NS; ++i) {
                const int r = i * RPIK + lane / CPRK;
                *reinterpret_cast<half8_t*>(&kt[r * D + (((lane % CPRK) ^ swz<D>(r)) << 3)]) = ka[i];
            }
#pragma unroll
            for (int ks = 0; ks < NS; ++ks)
                ka[ks] = *reinterpret_cast<const half8_t*>(&kt[c * D + (((2 * ks + h) ^ swz<D>(c)) << 3)]);
        }
    };
    // KNORM: the reciprocal root mean squares of a block's keys, through LDS from the lanes that hold the rows (lane and
    // lane^32 one half each) to the lanes that hold their scores
    __shared__ __attribute__((aligned(256))) float Kr[KNORM ? DNW * 32 : 4];
    float gk_unit = 1.f;       // the power of two that gamma_k was divided by
    auto key_norms = [&](const half8_t (&ka)[NS]) __attribute__((always_inline)) {
        float ss[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < NS; ++ks)
#pragma unroll
            for (int e = 0; e < 8; e += 2) {
                const half2_t p = {ka[ks][e], ka[ks][e + 1]};
                ss[e / 2] = __builtin_amdgcn_fdot2(p, p, ss[e / 2], false);
            }
        const float rstd = 1.0f / __builtin_sqrtf(half_sum((ss[0] + ss[1]) + (ss[2] + ss[3])) / (float)D + a.k_eps);
        Kr[wave * 32 + c] = rstd * gk_unit;                // (both lanes of a row write the same)
    };
    auto scale_scores = [&](float16_t& s) __attribute__((always_inline)) {
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4) {
            const float4_t w = *reinterpret_cast<const float4_t*>(&Kr[wave * 32 + 8 * r4 + 4 * h]);
#pragma unroll
            for (int e = 0; e < 4; ++e) s[r4 * 4 + e] *= w[e];
        }
    };
    // ---- V: block rows global -> LDS, chunk c of row r stored at c ^ swz<D>(r); load n covers rows n*RPI + lane/CPR
    const __amdgpu_buffer_rsrc_t vrs = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(a.v + b * a.vb + kvh * a.vh), 0, (int)(((int64_t)(a.Skv - 1) * a.vs + D) * 2), 0x00020000);
    int vvo[NI];
#pragma unroll
    for (int n = 0; n < NI; ++n) {
        const int r = n * RPI + lane / CPR;
        vvo[n] = (int)(r * a.vs * 2) + dsl * DV * 2 + (((lane % CPR) ^ swzv<DV>(r)) << 4);
    }
    const int vblk_bytes = (int)(32 * a.vs * 2);
#define TRN_FETCH_V(blk_, dst_)                                                                                  \
    _Pragma("unroll") for (int n_ = 0; n_ < NI; ++n_) __builtin_amdgcn_raw_ptr_buffer_load_lds(                  \
        vrs, (__attribute__((address_space(3))) void*)(&dst_[wave * 32 * DV + n_ * RPI * DV]), 16, vvo[n_],      \
        (blk_) * vblk_bytes, 0, 0)
    // V^T operand through the transposing read (as in the prefill kernel): rows 4h + (lane%16)/4 [+8] of a 16-key half
    int voff_lo[NDB], voff_hi[NDB];
    {
        const int rl = 4 * h + ((lane & 15) >> 2), rh = rl + 8;
        const int lc = 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1), sub = (lane & 1) * 4;
#pragma unroll
        for (int db = 0; db < NDB; ++db) {
            voff_lo[db] = wave * 32 * DV + rl * DV + (((db * 4 + lc) ^ swzv<DV>(rl)) << 3) + sub;
            voff_hi[db] = wave * 32 * DV + rh * DV + (((db * 4 + lc) ^ swzv<DV>(rh)) << 3) + sub;
        }
    }

    float16_t oacc[NDB];
#pragma unroll
    for (int i = 0; i < NDB; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[i][r] = 0.f;
    float m = -INFINITY, l = 0.f;       // running max (log2 domain, shared by the lane pair) and this lane's partial sum
    float m2 = -INFINITY, l2 = 0.f;     // the same for the perturbed scores (KeyFormer)
    // KeyFormer noise: this lane's query row, the 4 x 4 keys of its accumulator layout per block, one block ahead; kept as
    // it arrives (three dwords per 4 keys of fp16 noise) and widened where it is used, so that nothing waits for it here
    typedef typename std::conditional<N16, uint3_t, float4_t>::type noise_t;
    const void* nbase = NOISE ? reinterpret_cast<const char*>(a.noise) + (b * a.nb + head * a.nh) * (N16 ? 2 : 4) : nullptr;
    const HalfNoise hn(nbase, N16 ? a.Sq : 1, N16 ? a.ns : 0, N16 ? a.Skv : 0);
    const __amdgpu_buffer_rsrc_t nrs = N16 ? hn.rs : __builtin_amdgcn_make_buffer_rsrc(
        (void*)nbase, 0, NOISE ? (int)(((int64_t)(a.Sq - 1) * a.ns + a.Skv) * 4) : 0, 0x00020000);
    int nsh = 0;
    const int nvo = N16 ? hn.row((int64_t)qrow_ld * a.ns + 4 * h, nsh) : NOISE ? (int)(((int64_t)qrow_ld * a.ns + 4 * h) * 4) : 0;
    noise_t g0[4], g1[4];
    auto fetch_noise = [&](int blk, noise_t (&g)[4]) __attribute__((always_inline)) {
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4) {
            if constexpr (N16) g[r4] = __builtin_bit_cast(noise_t, __builtin_amdgcn_raw_buffer_load_b96(nrs, nvo + r4 * 16, blk * 64, 0));
            else g[r4] = __builtin_bit_cast(noise_t, __builtin_amdgcn_raw_buffer_load_b128(nrs, nvo + r4 * 32, blk * 128, 0));
        }
    };

    // this workgroup's blocks: a contiguous share of the keys when they are split over several workgroups
    int visible = a.Skv;                                // keys that some query of the tile sees
    if (a.causal) visible = min(visible, min(q0 + 31, a.Sq - 1) + off + 1);
    const int nblk_all = (visible + 31) / 32, bps = PARTS || NOISE || SWEEP ? (nblk_all + a.n_split - 1) / a.n_split : nblk_all;
    const int blk0 = split * bps, nblk = max(0, min(nblk_all, blk0 + bps) - blk0);
    const int nmine = nblk > wave ? (nblk - wave + DNW - 1) / DNW : 0;          // blocks blk0 + wave, + 8, ...
    half8_t ka0[NS], ka1[NS];
    const int q = tid & 31, dg = tid >> 5;                // merges: 16 groups of threads share out the DV/4 quads of a query
    const int bh = b * a.Hq + head;
    constexpr int KB = KEEP ? kept_blocks(D, DS, NOISE) : 1;
    float16_t kept[KB];
    float mstar = -INFINITY, L = 0.f, ms2 = -INFINITY, L2 = 0.f;      // of the merged partial results

    // One 32-key block whose K is in kc and whose V is in stage Vc; the next block's loads go to kn / Vn first.
    // keep (KEEP only): the block's scores in the log2 domain, the perturbed ones with noise, -inf where masked.
    auto block = [&](int it, half8_t (&kc)[NS], half8_t (&kn)[NS], const half_t* Vc, half_t* Vn, noise_t (&gc)[4],
                     noise_t (&gn)[4], float16_t& keep) __attribute__((always_inline)) {
        const int blk = blk0 + wave + it * DNW, key0 = blk * 32;
        // (with noise the registers are short: K is then single-buffered, refilled as soon as the scores are issued)
        if constexpr (!NOISE) fetch_k(blk + DNW, kn);
        if constexpr (!NOISE && VSINGLE) __builtin_amdgcn_sched_barrier(0);      // (in flight before this block's K is waited for)
        if constexpr (!VSINGLE) {
            // (Vn is the stage the previous block read: the same fence as for the single stage below, so that the order
            // does not hang on where the compiler happens to cut its scheduling regions)
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_waitcnt(0xc07f);        // lgkmcnt(0)
            TRN_FETCH_V(blk + DNW, Vn);
        }
        if constexpr (NOISE) fetch_noise(blk + DNW, gn);
        float16_t s;
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] = 0.f;
        k_operands(kc);
        if constexpr (KNORM) key_norms(kc);
#pragma unroll
        for (int ks = 0; ks < NS; ++ks) s = mfma32(kc[ks], qB[ks], s);
        if constexpr (KNORM) scale_scores(s);
        if constexpr (NOISE) fetch_k(blk + DNW, kc);
        // mask (wave-uniform test), block max, running max, probabilities
        const bool masked = (key0 + 32 > a.Skv) || (a.causal && key0 + 31 > q0 + off);
        if (masked) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int key = key0 + 8 * (r / 4) + 4 * h + (r % 4);
                s[r] = (key < a.Skv && (!a.causal || key <= qrow + off)) ? s[r] : -INFINITY;
            }
        }
        if constexpr (NOISE) {          // row normaliser of z = (scale*s + g)/tau in the log2 domain
            float16_t z;
#pragma unroll
            for (int r4 = 0; r4 < 4; ++r4) {
                if constexpr (N16) {
                    const half4_t gv = half_noise4(gc[r4], nsh);
#pragma unroll
                    for (int e = 0; e < 4; ++e) z[r4 * 4 + e] = __builtin_fmaf((float)gv[e], a.c3, s[r4 * 4 + e] * a.c2);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) z[r4 * 4 + e] = __builtin_fmaf(gc[r4][e], a.c3, s[r4 * 4 + e] * a.c2);
                }
            }
            if (masked) {               // a select, not arithmetic: what lies past a row's last key (the padding of
                                        // the noise pitch) may be anything, NaN included
#pragma unroll
                for (int r = 0; r < 16; ++r) z[r] = s[r] == -INFINITY ? -INFINITY : z[r];
            }
            if constexpr (KEEP) keep = z;
            const float zmax = fmaxf(m2, half_max(max16(z)));
            if (zmax > -INFINITY) {
                float sum = 0.f;
#pragma unroll
                for (int r = 0; r < 16; ++r) sum += fast_exp2(z[r] - zmax);
                l2 = l2 * fast_exp2(m2 - zmax) + sum;
                m2 = zmax;
            }
        }
        if constexpr (KEEP && !NOISE) {
#pragma unroll
            for (int r = 0; r < 16; ++r) keep[r] = s[r] == -INFINITY ? -INFINITY : s[r] * a.c1;
        }
        const float smax = half_max(max16(s)) * a.c1;
        const float mnew = fmaxf(m, smax);
        const float mref = mnew == -INFINITY ? 0.f : mnew;     // a row can see nothing of a block
        const float alpha = fast_exp2(m - mref);               // m = -inf: 0
        const half2_t ones = {(half_t)1.f, (half_t)1.f};
        half8_t pB[2];
        l *= alpha;
#pragma unroll
        for (int r = 0; r < 16; r += 2) {
            const half2_t pp = {(half_t)fast_exp2(__builtin_fmaf(s[r], a.c1, -mref)),
                                (half_t)fast_exp2(__builtin_fmaf(s[r + 1], a.c1, -mref))};
            l = __builtin_amdgcn_fdot2(pp, ones, l, false);    // the row sum of exactly the values that multiply V
            pB[r / 8][r % 8] = pp[0]; pB[r / 8][r % 8 + 1] = pp[1];
        }
#pragma unroll
        for (int i = 0; i < NDB; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) oacc[i][r] *= alpha;
        m = mnew;
        // this block's V has landed: behind it only the next block's NS + NI (+ 4 noise) requests were issued
        // (one V stage: its refill is issued behind the block's P V, so only K and noise requests are younger)
        constexpr int kBehind = NS + (VSINGLE ? 0 : NI) + (NOISE ? 4 : 0);
        __builtin_amdgcn_s_waitcnt(0x0f70 | (kBehind & 15) | ((kBehind >> 4) << 14));
#pragma unroll
        for (int i = 0; i < NSV; ++i) {
            const half_t* vp = Vc + 16 * (i / NDB) * DV;
            const half4_t lo = lds_read_tr16(vp + voff_lo[i % NDB]);
            const half4_t hi = lds_read_tr16(vp + voff_hi[i % NDB]);
            const half8_t va = half8_t{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
            oacc[i % NDB] = mfma32(va, pB[i / NDB], oacc[i % NDB]);
        }
        // (The refill must not overtake the stage's readers.  The compiler does not order the global->LDS load
        // behind the transposing reads by itself -- left alone it moved the load in front of the last of them -- hence
        // the scheduling fence; the wait makes the reads' return explicit.)
        if constexpr (VSINGLE) {
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_waitcnt(0xc07f);        // lgkmcnt(0)
            TRN_FETCH_V(blk + DNW, Vn);
        }
    };
    if constexpr (!SWEEP) {
    fetch_k(blk0 + wave, ka0);
    TRN_FETCH_V(blk0 + wave, Vs0);
    if constexpr (NOISE) fetch_noise(blk0 + wave, g0);
    // (the first K / V requests are on their way before Q is waited for: one memory latency instead of two)
    if (a.q_norm || KNORM) {
        if constexpr (KNORM) {
            // gamma_k over the power of two above its largest element, so that no query grows by it
            float top = 0.f;
#pragma unroll
            for (int ks = 0; ks < NS; ++ks) {
#pragma unroll
                for (int e = 0; e < 8; ++e) top = fmaxf(top, __builtin_fabsf((float)gk[ks][e]));
            }
            top = half_max(top);
            if (top > 0.f && top < INFINITY) gk_unit = __builtin_ldexpf(1.f, __builtin_amdgcn_frexp_expf(top));
        }
        float rstd = 1.f;
        if (a.q_norm) {
            float ss = 0.f;
#pragma unroll
            for (int ks = 0; ks < NS; ++ks)
#pragma unroll
                for (int e = 0; e < 8; ++e) { float f = (float)qB[ks][e]; ss += f * f; }
            ss = half_sum(ss);
            rstd = 1.0f / __builtin_sqrtf(ss / (float)D + a.q_eps);
        }
        const float per_unit = 1.f / gk_unit;
#pragma unroll
        for (int ks = 0; ks < NS; ++ks) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                float y = (float)qB[ks][e] * rstd;
                if (use_gq) y = (float)gq[ks][e] * y;
                if constexpr (KNORM) y *= (float)gk[ks][e] * per_unit;
                qB[ks][e] = (half_t)y;
            }
        }
    }
    // pin the arrival of Q here: left to the first MFMA in the loop, the compiler's wait would sit in the loop body
#pragma unroll
    for (int ks = 0; ks < NS; ++ks) asm volatile("" ::"v"(qB[ks]));
    auto even = [&](int it, float16_t& keep) __attribute__((always_inline)) {
        if constexpr (NOISE) block(it, ka0, ka0, Vs0, VSINGLE ? Vs0 : Vs1, g0, g1, keep);
        else block(it, ka0, ka1, Vs0, VSINGLE ? Vs0 : Vs1, g0, g1, keep);
    };
    auto odd = [&](int it, float16_t& keep) __attribute__((always_inline)) {
        if constexpr (NOISE) block(it, ka0, ka0, VSINGLE ? Vs0 : Vs1, Vs0, g1, g0, keep);
        else block(it, ka1, ka0, VSINGLE ? Vs0 : Vs1, Vs0, g1, g0, keep);
    };
    if constexpr (KEEP) {
        // (nested, so that a block's waits are sized on one path only)
        auto walk = [&](auto&& self, auto at) __attribute__((always_inline)) {
            constexpr int it = decltype(at)::value;
            if constexpr (it < KB) {
                if (it < nmine) {
                    if constexpr (it % 2 == 0) even(it, kept[it]); else odd(it, kept[it]);
                    self(self, std::integral_constant<int, it + 1>{});
                }
            }
        };
        walk(walk, std::integral_constant<int, 0>{});
    } else {
        for (int it = 0; it < nmine; it += 2) {
            even(it, kept[0]);
            if (it + 1 < nmine) odd(it + 1, kept[0]);
        }
    }
#undef TRN_FETCH_V

    // ---- merge the eight waves' (m, l, O^T) through LDS.  Partial O^T as float4 quads [d/4][query]: the first half
    // of the columns in this wave's part of Vs0, the second half in its part of Vs1 (each exactly 32 * DV/2 floats).
    half_t* const Vhi = VSINGLE ? Kt : Vs1;            // (one V stage: the K area, as large, takes the second half)
    l = half_sum(l);
    __builtin_amdgcn_s_waitcnt(0x0f70);                 // the look-ahead requests past the end have landed too
    if (h == 0) { st_m[wave][c] = m; st_l[wave][c] = l; }
    if constexpr (NOISE) {
        l2 = half_sum(l2);
        if (h == 0) { st_m2[wave][c] = m2; st_l2[wave][c] = l2; }
    }
#pragma unroll
    for (int db = 0; db < NDB; ++db) {
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4) {
            const int quad = db * 8 + 2 * r4 + h;             // columns 4 quad .. +3 of this workgroup's share
            float4_t* part = reinterpret_cast<float4_t*>((quad < DV / 8 ? Vs0 : Vhi) + wave * 32 * DV);
            part[(quad % (DV / 8)) * 32 + c] =
                float4_t{oacc[db][r4 * 4], oacc[db][r4 * 4 + 1], oacc[db][r4 * 4 + 2], oacc[db][r4 * 4 + 3]};
        }
    }
    __syncthreads();
    constexpr int NQD = (DV / 4 + 15) / 16;               // quads per thread (with 8 quads, half the groups have none)
    mstar = st_m[0][q];
#pragma unroll
    for (int w = 1; w < DNW; ++w) mstar = fmaxf(mstar, st_m[w][q]);
    float4_t acc[NQD];
    {
        float wgt[DNW];
#pragma unroll
        for (int w = 0; w < DNW; ++w) {                   // idle waves: m = -inf, weight 0
            wgt[w] = mstar == -INFINITY ? 0.f : fast_exp2(st_m[w][q] - mstar);
            L += st_l[w][q] * wgt[w];
        }
#pragma unroll
        for (int qi = 0; qi < NQD; ++qi) {
            const int quad = min(dg + 16 * qi, DV / 4 - 1);   // d = 4*quad .. +3 (a group without a quad re-reads the last)
            const half_t* base = quad < DV / 8 ? Vs0 : Vhi;
            const int ql = quad % (DV / 8);
            acc[qi] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int w = 0; w < DNW; ++w) acc[qi] += reinterpret_cast<const float4_t*>(base + w * 32 * DV)[ql * 32 + q] * wgt[w];
        }
    }
    if constexpr (NOISE) {
#pragma unroll
        for (int w = 0; w < DNW; ++w) ms2 = fmaxf(ms2, st_m2[w][q]);
#pragma unroll
        for (int w = 0; w < DNW; ++w) L2 += ms2 == -INFINITY ? 0.f : st_l2[w][q] * fast_exp2(st_m2[w][q] - ms2);
    }
    if (DS == 1 && (PARTS || (NOISE && !KEEP && a.n_split > 1))) {
        // ---- keys split over workgroups: publish (m, l, unnormalised O) of this share; the next launch merges all shares or, in one launch
        // with score perturbation, the workgroup that arrives last at the head's counter.  Workspace: [arrival counters, 256-byte aligned][bh][split] (two launches: without the counters)
        // {O as quads [D/4][32 queries][4], (m, l, m2, l2) [32]} floats.  The shares travel as device-scope atomic stores and loads, which
        // go to the memory all L2 slices agree on (a fence that makes ordinary stores visible writes back and
        // invalidates a whole L2, and with one per wave that took several times the kernel's own time); the arrival
        // is a release/acquire increment by ONE thread, tied to the other threads by the workgroup barriers.
        constexpr int PART = 32 * (D + 4);
        const int n_bh = a.B * a.Hq;
        unsigned* counters = reinterpret_cast<unsigned*>(a.ws);
        float* parts = !NOISE || a.partial ? a.ws : a.ws + ((n_bh + 63) / 64) * 64;
        const bool query = q < a.Sq;
        if (!NOISE || a.partial) {             // (the merge is the next launch's: ordinary stores)
            float* p = parts + ((int64_t)bh * a.n_split + split) * PART;
            if (a.partial == 2 && !query) return;
#pragma unroll
            for (int qi = 0; qi < NQD; ++qi) *reinterpret_cast<float4_t*>(p + ((dg + 16 * qi) * 32 + q) * 4) = acc[qi];
            if (dg == 0) *reinterpret_cast<float4_t*>(p + 32 * D + 4 * q) = float4_t{mstar, L, ms2, L2};
            return;
        }
        float* mine = parts + ((int64_t)bh * a.n_split + split) * PART;
        auto publish = [](float* p, float4_t v) __attribute__((always_inline)) {
            const ulong2_t u = __builtin_bit_cast(ulong2_t, v);
            __hip_atomic_store(reinterpret_cast<unsigned long long*>(p), u[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(reinterpret_cast<unsigned long long*>(p) + 1, u[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        };
        auto collect = [](const float* p) __attribute__((always_inline)) {
            ulong2_t u;
            u[0] = __hip_atomic_load(reinterpret_cast<const unsigned long long*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            u[1] = __hip_atomic_load(reinterpret_cast<const unsigned long long*>(p) + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return __builtin_bit_cast(float4_t, u);
        };
        if (query) {
#pragma unroll
            for (int qi = 0; qi < NQD; ++qi) publish(mine + ((dg + 16 * qi) * 32 + q) * 4, acc[qi]);
            if (dg == 0) publish(mine + 32 * D + 4 * q, float4_t{mstar, L, ms2, L2});
        }
        __syncthreads();                                   // every wave's stores have been acknowledged
        __shared__ unsigned arrival;
        // (release/acquire at device scope makes the hand-over of the shares hold by the memory model alone -- the other
        // threads' stores are ordered before it by the workgroup barrier; it costs one L2 write-back and one invalidate
        // per WORKGROUP, about 1.5 us per launch)
        if (tid == 0) arrival = __hip_atomic_fetch_add(&counters[bh], 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (arrival != (unsigned)(a.n_split - 1)) return;
        const float* head_parts = parts + (int64_t)bh * a.n_split * PART;
        // shares are fetched eight at a time (all requests of a batch in flight together) and folded in with a
        // running maximum, in share order: the result does not depend on which workgroup does the merge
        mstar = -INFINITY; ms2 = -INFINITY; L = 0.f; L2 = 0.f;
#pragma unroll
        for (int qi = 0; qi < NQD; ++qi) acc[qi] = float4_t{0.f, 0.f, 0.f, 0.f};
        constexpr int BATCH = 8;
        for (int s0 = 0; query && s0 < a.n_split; s0 += BATCH) {
            float4_t st[BATCH], d[BATCH][NQD];
#pragma unroll
            for (int u = 0; u < BATCH; ++u) {
                const float* ps = head_parts + min(s0 + u, a.n_split - 1) * PART;
                st[u] = collect(ps + 32 * D + 4 * q);
#pragma unroll
                for (int qi = 0; qi < NQD; ++qi) d[u][qi] = collect(ps + ((dg + 16 * qi) * 32 + q) * 4);
            }
#pragma unroll
            for (int u = 0; u < BATCH; ++u) {
                if (s0 + u >= a.n_split) break;
                const float mnew = fmaxf(mstar, st[u][0]);
                if (mnew > -INFINITY) {                        // -inf: a share that saw no key of this query
                    const float wa = fast_exp2(mstar - mnew), wb = fast_exp2(st[u][0] - mnew);
                    L = L * wa + st[u][1] * wb;
#pragma unroll
                    for (int qi = 0; qi < NQD; ++qi) acc[qi] = acc[qi] * wa + d[u][qi] * wb;
                    mstar = mnew;
                }
                if constexpr (NOISE) {
                    const float m2new = fmaxf(ms2, st[u][2]);
                    if (m2new > -INFINITY) {
                        L2 = L2 * fast_exp2(ms2 - m2new) + st[u][3] * fast_exp2(st[u][2] - m2new);
                        ms2 = m2new;
                    }
                }
            }
        }
        if (tid == 0) __hip_atomic_store(&counters[bh], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);                   // left as found: the next launch on the stream starts from zero
    }
    {
        const float inv = 1.0f / L;
        half_t* orow = a.o + b * a.ob + head * a.oh + (int64_t)(q0 + q) * a.os + dsl * DV;
        if (q0 + q < a.Sq) {
#pragma unroll
            for (int qi = 0; qi < NQD; ++qi) {
                const half4_t ov = {(half_t)(acc[qi][0] * inv), (half_t)(acc[qi][1] * inv), (half_t)(acc[qi][2] * inv), (half_t)(acc[qi][3] * inv)};
                if (dg + 16 * qi < DV / 4) *reinterpret_cast<half4_t*>(orow + 4 * (dg + 16 * qi)) = ov;
            }
        }
        // (every column share holds the same row normalisers: the first one writes them)
        if (dg == 0 && dsl == 0 && q0 + q < a.Sq && a.lse) a.lse[(int64_t)bh * a.Sq + q0 + q] = (mstar + fast_log2(L)) * kLn2;
        if constexpr (NOISE) {
            if (dg == 1 && dsl == 0 && q0 + q < a.Sq) a.lse_pert[(int64_t)bh * a.Sq + q0 + q] = (ms2 + fast_log2(L2)) * kLn2;
        }
    }
    } else {
        // ---- the launch behind a.partial: every workgroup of a head merges the row normalisers of all its shares, each a
        // part of the output columns, and sweeps over its own share of the keys below
        constexpr int PART = 32 * (D + 4), BATCH = 8;
        const float* parts = a.ws + (int64_t)bh * a.n_split * PART;
        const int quads = (D / 4 + a.n_split - 1) / a.n_split, quad = split * quads + dg;     // at most 16: two shares or more
        const bool merges = dg < quads && quad < D / 4;
        const float* op = parts + (min(quad, D / 4 - 1) * 32 + q) * 4;
        float4_t d[BATCH];
        auto fetch_o = [&](int s0) __attribute__((always_inline)) {
#pragma unroll
            for (int u = 0; u < BATCH; ++u) d[u] = *reinterpret_cast<const float4_t*>(op + min(s0 + u, a.n_split - 1) * PART);
        };
        if (merges) fetch_o(0);
        float4_t* const st = reinterpret_cast<float4_t*>(Kt);            // [share][query]: 16 KB for kMaxStatSplits
        for (int s = dg; s < a.n_split; s += 16) st[s * 32 + q] = *reinterpret_cast<const float4_t*>(parts + s * PART + 32 * D + 4 * q);
        __syncthreads();
        for (int s = 0; s < a.n_split; ++s) { mstar = fmaxf(mstar, st[s * 32 + q][0]); ms2 = fmaxf(ms2, st[s * 32 + q][2]); }
        for (int s = 0; s < a.n_split; ++s) {
            const float4_t v = st[s * 32 + q];
            if (mstar > -INFINITY) L += v[1] * fast_exp2(v[0] - mstar);
            if (NOISE && ms2 > -INFINITY) L2 += v[3] * fast_exp2(v[2] - ms2);
        }
        if (merges) {
            float4_t o = {0.f, 0.f, 0.f, 0.f};
            for (int s0 = 0; s0 < a.n_split; s0 += BATCH) {
                if (s0 > 0) fetch_o(s0);
#pragma unroll
                for (int u = 0; u < BATCH; ++u)
                    if (s0 + u < a.n_split && mstar > -INFINITY) o += d[u] * fast_exp2(st[(s0 + u) * 32 + q][0] - mstar);
            }
            const float inv = 1.0f / L;
            const half4_t ov = {(half_t)(o[0] * inv), (half_t)(o[1] * inv), (half_t)(o[2] * inv), (half_t)(o[3] * inv)};
            if (q < a.Sq) *reinterpret_cast<half4_t*>(a.o + b * a.ob + head * a.oh + (int64_t)q * a.os + 4 * quad) = ov;
        }
        if (split == 0 && dg == 0 && q < a.Sq) {
            if (a.lse) a.lse[(int64_t)bh * a.Sq + q] = (mstar + fast_log2(L)) * kLn2;
            if constexpr (NOISE) a.lse_pert[(int64_t)bh * a.Sq + q] = (ms2 + fast_log2(L2)) * kLn2;
        }
    }
    // ---- column statistics (KeyFormer key scores, RoCo sums), from the kept scores or by a second sweep over this head's keys now that the
    // row normalisers are final.  The score block is formed the other way round, S[query][key] -- the same two
    // register operands with their roles swapped -- so that a lane owns one KEY and holds 16 of the 32 queries: the
    // sum over queries is in-lane plus one exchange with lane^32, and a block's 32 sums are one 128-byte store.
    // (One query tile only.  Not with the keys split over workgroups -- the statistics need the normalisers of the whole head; the column
    // shares of a head all have them, and take every DS-th round of blocks of the sweep each.)
    if constexpr (KEEP) {
        __syncthreads();                                   // every thread has read the merge arrays
        if (dg == 0) st_l[0][q] = NOISE ? ms2 + fast_log2(L2) : mstar + fast_log2(L);     // log2 domain
        __syncthreads();
        const float lq = c < a.Sq ? st_l[0][c] : INFINITY;       // (lanes without a query add nothing)
        // 4 KB of this wave's own for the sums of a block and, in two halves, for those of its squares
        float* const area = reinterpret_cast<float*>(Kt) + wave * (D * 16);
        float* const sq_lo = D == 128 ? area + 1024 : reinterpret_cast<float*>(Vs0) + wave * (DV * 16);
        float* const sq_hi = D == 128 || DV == 64 ? sq_lo + 512 : reinterpret_cast<float*>(Vs1) + wave * (DV * 16);
#pragma unroll
        for (int it = 0; it < KB; ++it) {
            if (it >= nmine || it % DS != dsl) continue;         // (the column shares take every DS-th block each)
            float p[16], x, y = 0.f;
#pragma unroll
            for (int r = 0; r < 16; ++r) p[r] = kept[it][r] == -INFINITY ? 0.f : fast_exp2(kept[it][r] - lq);
            put_sums(p, area, area + 512, lane);
            if (a.col_sumsq) {
#pragma unroll
                for (int r = 0; r < 16; ++r) p[r] *= p[r];
                put_sums(p, sq_lo, sq_hi, lane);
                x = key_sum(area, area + 512, lane);
                y = key_sum(sq_lo, sq_hi, lane);
            } else x = key_sum(area, area + 512, lane);
            const int key = (blk0 + wave + it * DNW) * 32 + key_of_sum(lane);
            if ((lane & 1) == 0 && key < a.Skv) {
                const int64_t at = (int64_t)bh * a.Skv + key;
                store_stat(a.col_sum, a.s16, at, x);
                store_stat(a.col_sumsq, a.s16, at, y);
            }
        }
    } else if (!KNORM && (a.col_sum || a.col_sumsq || a.probs)) {
        __syncthreads();                                   // every thread has read the merge arrays
        if (dg == 0) st_l[0][q] = NOISE ? ms2 + fast_log2(L2) : mstar + fast_log2(L);     // log2 domain
        __syncthreads();
        float lq[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) lq[r] = st_l[0][8 * (r / 4) + 4 * h + (r % 4)];
        const float cs = NOISE ? a.c2 : a.c1;
        // noise of the lane's key for its 16 queries: 16 dwords from 16 rows, consecutive keys in consecutive lanes
        float gs0[NOISE ? 16 : 1], gs1[NOISE ? 16 : 1];
        auto fetch_noise_col = [&](int blk, float (&g)[NOISE ? 16 : 1]) __attribute__((always_inline)) {
            if constexpr (NOISE) {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int qr = 8 * (r / 4) + 4 * h + (r % 4);
                    if constexpr (N16)
                        g[r] = (float)__builtin_bit_cast(half_t, __builtin_amdgcn_raw_buffer_load_b16(
                            nrs, (int)((qr * a.ns + c + hn.odd) * 2), blk * 64, 0));
                    else
                        g[r] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                            nrs, (int)((qr * a.ns + c) * 4), blk * 128, 0));
                }
            }
        };
        // (one block ahead is enough: with one workgroup per head the sweep runs at what a single CU can pull from
        // L2, about 55 GB/s; requesting two blocks ahead measured the same)
        auto sweep = [&](int it, half8_t (&kc)[NS], half8_t (&kn)[NS], float (&gc)[NOISE ? 16 : 1], float (&gn)[NOISE ? 16 : 1])
                         __attribute__((always_inline)) {
            const int blk = blk0 + dsl * DNW + wave + it * DNW * DS, key = blk * 32 + c;
            fetch_k(blk + DNW * DS, kn);
            fetch_noise_col(blk + DNW * DS, gn);
            float16_t s;
#pragma unroll
            for (int r = 0; r < 16; ++r) s[r] = 0.f;
            k_operands(kc);
#pragma unroll
            for (int ks = 0; ks < NS; ++ks) s = mfma32(qB[ks], kc[ks], s);
            float x = 0.f, y = 0.f;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int qr = 8 * (r / 4) + 4 * h + (r % 4);
                float t = __builtin_fmaf(s[r], cs, -lq[r]);
                if constexpr (NOISE) t = __builtin_fmaf(gc[r], a.c3, t);
                const bool ok = key < a.Skv && qr < a.Sq && (!a.causal || key <= qr + off);
                const float p = ok ? fast_exp2(t) : 0.f;
                // (32 consecutive keys of one query row per store instruction: whole 128-byte lines)
                if (a.probs && key < a.Skv && qr < a.Sq) a.probs[((int64_t)bh * a.Sq + qr) * a.Skv + key] = p;
                x += p;
                y = __builtin_fmaf(p, p, y);
            }
            x = half_sum(x); y = half_sum(y);
            // (the statistics kernels' other form: the second launch has every query's probabilities of its keys too)
            if constexpr (SWEEP && !NOISE) {
                if (a.mean_std) mean_std_of(x, y, (float)(a.causal ? a.Sq - max(0, key - off) : a.Sq));
            }
            if (h == 0 && key < a.Skv) {
                const int64_t at = (int64_t)bh * a.Skv + key;
                store_stat(a.col_sum, a.s16, at, x);
                store_stat(a.col_sumsq, a.s16, at, y);
            }
        };
        const int first = dsl * DNW + wave;
        const int nsweep = nblk > first ? (nblk - first + DNW * DS - 1) / (DNW * DS) : 0;
        fetch_k(blk0 + first, ka0);
        fetch_noise_col(blk0 + first, gs0);
        for (int it = 0; it < nsweep; it += 2) {
            sweep(it, ka0, ka1, gs0, gs1);
            if (it + 1 < nsweep) sweep(it + 1, ka1, ka0, gs1, gs0);
        }
    }
#endif
}

// Arrival counters, and the shares' partial results behind them.
static int64_t counter_bytes(int64_t n_bh) { return (n_bh + 63) / 64 * 256; }
static int64_t share_bytes(int64_t n_bh, int ns, int head_dim) { return n_bh * ns * 32 * (head_dim + 4) * 4; }
static int64_t split_bytes(int64_t n_bh, int ns, int head_dim) { return ns <= 1 ? 0 : counter_bytes(n_bh) + share_bytes(n_bh, ns, head_dim); }
int64_t attn_decode_workspace_bytes(int batch, int n_q_heads, int seq_q, int seq_kv, int head_dim) {
    if (seq_q > 32) return 0;
    const int ns = decode_splits(batch * n_q_heads, seq_kv);
    if (ns <= 1) return 0;
    const int64_t n_bh = (int64_t)batch * n_q_heads;
    return split_bytes(n_bh, ns, head_dim);
}

// The shares' partial results alone, of two launches below that rule's lines: behind as many bytes as the counters of any number of heads that has
// some take, so that a workspace with counters in it serves these calls too.
constexpr int kCounterRoom = 512;
int64_t attn_few_query_workspace_bytes(int batch, int n_q_heads, int n_kv_heads, int seq_q, int seq_kv, int head_dim) {
    if (seq_q > 32 || decode_splits(batch * n_q_heads, seq_kv) > 1) return 0;
    const int ns = few_query_shares(batch * n_q_heads, batch * n_kv_heads, seq_kv, head_dim);
    return ns > 1 ? kCounterRoom + share_bytes((int64_t)batch * n_q_heads, ns, head_dim) : 0;
}

// Column shares of a head for `units` = heads x query tiles: as many as leave 32 columns per workgroup and at most one
// workgroup per CU.  (Two per CU do not fit, and a second round costs what the first did: 128 units of head_dim 128, us
// 1 / 2 / 4 shares: 400 keys 10.3 / 8.7 / 13.7, 4100 keys 34 / 26 / 45.)
static int decode_col_shares(int64_t units, int seq_q, int seq_kv, int head_dim) {
    int ds = 1;
    if (seq_kv >= 256 || seq_q > 32)
        while (ds < 4 && head_dim / (ds * 2) >= 32 && units * ds * 2 <= 256) ds *= 2;
    return ds;
}

// More than 32 queries per head: tiles of 32 queries, eight waves sharing out the keys of each, against the prefill
// kernels' 128-query workgroups whose waves walk all the keys -- better as long as the tiles are no more than the CUs,
// i.e. while the prefill kernels would leave most of the chip idle.  Measured, us prefill / here: 32 heads of 128: 100
// queries on 4100 keys 63 / 26, on 400 12.6 / 8.7, causal 256 on 256 10.6 / 8.9 (256 tiles), causal 350 on 350 12.3 / 14.4
// (352 tiles); 8 heads of 128, causal 777 on 777 17.6 / 12.2; 71 heads of 64: 64 queries on 4064 keys 41 / 19.  With more
// tiles than CUs: head_dim 64 on long caches (71 heads, 100 queries: 4100 keys 42 / 35, 1124 keys 15.6 / 15.6, 164 keys
// 6.8 / 10.2); with score perturbation, where the prefill kernel is slower, any (32 heads of 128, causal 350 on 350 22 /
// 19; 71 heads of 64, 128 queries on 4128 keys 114 / 83; but 781 tiles 20 / 25).
// Few heads of 128 under a causal mask have long tiles, which come first, and the CUs of the short ones take those past 256:
// us, split keys (narrow workgroups below 1100 keys) / here: one head of 4: 2071 keys (260 tiles) 24.1 / 19.6, 2807 30.0 / 24.7, 3575 (448) 35.6 / 33.6, 4055
// (508) 39.6 / 39.5; of 8: 1143 (288) 17.3 / 14.5, 1399 19.4 / 18.2, 1591 (400) 21.2 / 20.9, 1783 22.4 / 22.8; of 10: 823 (260) 15.4 / 12.9,
// 1015 18.5 / 16.4, 1111 (350) 17.8 / 17.5, 1271 18.7 / 19.2; of 12: 727 (276) 15.0 / 13.8, 855 (324) 16.7 / 15.4; of 14: 695 (308) 14.0 / 14.1; of 16: 567 (288) 12.3 / 13.1.
// (Not the attention that adds the sums of KeyFormer's single pass: this launch does not.)
bool attn_decode_suits(int batch, int n_q_heads, int seq_q, int seq_kv, int head_dim, bool causal, bool noise) {
    if (seq_q <= 32) return true;
    const int64_t bh = (int64_t)batch * n_q_heads, tiles = bh * ((seq_q + 31) / 32);
    if (head_dim == 128 && causal && seq_q == seq_kv && bh <= 12 && tiles <= (bh <= 4 ? 448 : bh <= 8 ? 400 : bh <= 10 ? 350 : 330)) return true;
    return tiles <= 256 || (tiles < 512 && (noise || (head_dim == 64 && seq_kv >= 1024)));
}

// Each tile of 32 queries normalises the keys it reads, some 0.25 us per 256 keys against 3 - 5 us for a launch: up to 2048.
// us, launch / here: 8 heads of 128, 1024 tokens 18.5 / 17.0; 2 x 8, 394 14.0 / 11.9.  (Not where a CU has a second tile of head_dim 128:
// 8 heads, 1399 22.9 / 25.5; 10, 1015 21.0 / 23.0.)
bool attn_decode_norms_keys(int batch, int n_q_heads, int seq_q, int seq_kv, int head_dim) {
    return attn_decode_suits(batch, n_q_heads, seq_q, seq_kv, head_dim, false, false) && seq_kv <= 2048;
}

// Whether the scores of a head's keys fit the registers of one workgroup, for key statistics without a second sweep.
static bool decode_keeps(int batch, int n_q_heads, int seq_q, int seq_kv, int head_dim, bool noise) {
    const int ds = decode_col_shares((int64_t)batch * n_q_heads, seq_q, seq_kv, head_dim);
    return seq_q <= 32 && (seq_kv + 31) / 32 <= kept_blocks(head_dim, ds, noise) * DNW;
}

// Where the query tiles of a head go.  On one XCD they share K and V in its L2, but fewer than eight heads, or a number that
// leaves the last eight short, then leave XCDs idle: from the point where the others have more than a workgroup per CU the
// tiles are dealt to all eight instead.  us, together / spread: one head of 128, 845 queries and keys 30.0 / 9.3, 3213 132 /
// 24, causal 4097 83 / 32; two of 64, causal 5219 68 / 24; four of 128, causal 1529 26.9 / 21.5; twelve of 64, causal 1132 with
// noise 26.0 / 19.4; but four of 128, 35 queries on 9587 keys (8 workgroups per XCD) 62.0 / 66.3.
static bool decode_spread(int64_t n_bh, int n_qtiles, int ds) {
    const int64_t heads8 = (n_bh + 7) / 8;
    return n_qtiles > 1 && heads8 * 64 > 9 * n_bh && heads8 * n_qtiles * ds > 32;
}

// Key shares of a problem with key statistics, for the two launches; 0: the statistics are part of the one launch, which runs
// on one workgroup per head and column share.  The second launch and what the first hands to it cost 4 - 6 us.  us one launch /
// two, 8 (32) queries with fp16 noise; without: 16 heads of 64, 1600 keys 17.4 / 14.3 (20.6 / 15.9); 12.7 / 12.4, 2064 20.5 / 14.4
// (22.5 / 15.8); 15.5 / 12.9, 16400 127 / 31 (163 / 37); 103 / 29; 8 heads of 128, 1600 17.8 / 17.0 (22.0 / 20.0); 14.3 / 15.1, 4112
// 32.8 / 18.9 (39.0 / 21.9); 27.4 / 17.6; 32 heads of 128, 2064 21.5 / 25.3 (24.6 / 28.8); 17.3 / 23.4, 4112 40.8 / 35.0 (49.7 /
// 42.4); 34.6 / 33.1, 16400 152 / 83 (185 / 94); 136 / 79; 71 of 64, 2064 21.0 / 21.4 (27.2 / 25.3); 16.3 / 19.1, 4112 40.3 / 31.5
// (50.0 / 37.5); 33.9 / 29.3; 64 of 128, 4112 49.9 / 48.2 (59.5 / 58.1); 43.5 / 46.5, 8208 92.9 / 84.9; 82.9 / 78.6.
constexpr int kMaxStatSplits = 32;
static int stats_splits(int batch, int n_q_heads, int seq_q, int seq_kv, int head_dim, bool noise) {
    const int64_t n_bh = (int64_t)batch * n_q_heads, per_key = n_bh * head_dim;
    const int nblk = (seq_kv + 31) / 32;
    const int from = n_bh <= 16 ? (noise ? 1537 : 2048) : per_key <= 5120 ? (noise ? 3072 : 3712) : 8192;
    if (seq_q > 32 || n_bh > 128 || seq_kv < from) return 0;
    const int ns = max(1, min(min(kMaxStatSplits, (int)(256 / n_bh)), nblk / 8));
    const int bps = (nblk + ns - 1) / ns, n = (nblk + bps - 1) / bps;
    return n > 1 ? n : 0;
}
int64_t attn_decode_stats_workspace_bytes(int batch, int n_q_heads, int seq_q, int seq_kv, int head_dim, bool noise) {
    return split_bytes((int64_t)batch * n_q_heads, stats_splits(batch, n_q_heads, seq_q, seq_kv, head_dim, noise), head_dim);
}
// ... that a workspace holds: with the plain attention's, as many as that has; but sixteen at most -- 24 of up to 10 heads on long caches --, and not many
// more than 192 that read keys of their own, of 3 to 32 heads.  us of a decode step of one token, as many as stats_splits() / 24 / 16 / 12 / 8 / 6 / 4: KeyFormer, 8
// heads of 128: 4500 keys (32) 23.1 / 23.2 / 23.1 / 23.4, 10000 33.0 / 29.9 / 28.4 / 29.6, 15000 37.9 / 34.1 / 34.1 / 36.3; 16 of 64 (16): 4500 21.4 / - / - / 19.9 / 20.6, 15000
// 32.6 / - / - / 32.3 / 34.1; 32 of 128 (8): 3200 51.0 / - / - / - / - / 47.5 / 47.0, 10000 76.0 / - / - / - / - / 73.8 / 73.4; RoCo, 8 of 128: 10000 32.6 / 29.0 / 27.2 / 28.1 / 31.3.
// Of the two launches alone: 8 of 128 on 2, 19989 25.1 / 25.4 / 29.4 / 34.6, 5 of 128, 15891 28.7 / 29.3 / 32.2, 9 of 64 on one, 23227 25.2 / 24.4 / 28.0, 3 of 128, 11471 22.4 /
// 21.8 / 23.4; 26 of 64, 22142 49.5 / - / - / - / 49.9 / 53.4, 28 of 64, 13191 40.1 / - / - / - / 38.5 / 42.2; 17 of 64, 21902 37.0 / - / - / 36.5 / 41.8.
// Left out: 2 of 128, KeyFormer, 10000 22.3 / - / 23.2; 4, 15000 27.2 / - / 30.7; 40 of 64 (6 / 4 shares), 10000 45.8 / 47.5.
int attn_decode_stat_shares(int batch, int n_q_heads, int n_kv_heads, int seq_q, int seq_kv, int head_dim, bool noise, int64_t workspace_bytes) {
    if (seq_q > 32) return 0;
    const int nblk = (seq_kv + 31) / 32;
    for (const int ns : {stats_splits(batch, n_q_heads, seq_q, seq_kv, head_dim, noise), decode_splits(batch * n_q_heads, seq_kv)})
        if (ns > 1 && split_bytes((int64_t)batch * n_q_heads, ns, head_dim) <= workspace_bytes) {
            const int n_bh = batch * n_q_heads, n_bkv = batch * n_kv_heads;
            int cap = ns;
            if (n_bh > 10 && n_bkv <= 32) cap = min(16, max((seq_kv >= 10000 ? 208 : 192) / n_bkv, head_dim == 64 ? 8 : 1));
            else if (n_bh > 2 && n_bh <= 10 && (n_bh > 4 || seq_kv < 12000)) cap = seq_kv >= (n_bh <= 4 ? 9000 : 11000) ? 24 : 16;
            const int n = min(ns, cap), bps = (nblk + n - 1) / n;
            return (nblk + bps - 1) / bps;
        }
    return 0;
}

// Name of the instantiation launched for a problem without a workspace (a measurement aid: what a kernel trace shows).
const char* attn_decode_kernel_name(int batch, int n_q_heads, int seq_q, int seq_kv, int head_dim, bool noise) {
    const int ds = decode_col_shares((int64_t)batch * n_q_heads * ((seq_q + 31) / 32), seq_q, seq_kv, head_dim);
    if (head_dim == 128) {
        if (ds == 4) return noise ? "trn::attn_decode_kernel<128, 4, 1>" : "trn::attn_decode_kernel<128, 4, 0>";
        if (ds == 2) return noise ? "trn::attn_decode_kernel<128, 2, 1>" : "trn::attn_decode_kernel<128, 2, 0>";
        return noise ? "trn::attn_decode_kernel<128, 1, 1>" : "trn::attn_decode_kernel<128, 1, 0>";
    }
    if (ds == 2) return noise ? "trn::attn_decode_kernel<64, 2, 1>" : "trn::attn_decode_kernel<64, 2, 0>";
    return noise ? "trn::attn_decode_kernel<64, 1, 1>" : "trn::attn_decode_kernel<64, 1, 0>";
}

// The shares' results of a head's queries, added up, the second of two launches: a thread has four columns of one query, whose shares
// are requested eight at a time, and the launch is two memory latencies, 2.6 - 3 us.
template <int D>
__global__ __launch_bounds__(256) void attn_decode_merge_kernel(const AttnArgs a) {
    constexpr int PART = 32 * (D + 4), BATCH = 8;
    const int bh = blockIdx.x / (D / 32), q = threadIdx.x & 31, quad = (int)(blockIdx.x % (D / 32)) * 8 + (threadIdx.x >> 5);
    if (q >= a.Sq) return;
    const float* const parts = a.ws + (int64_t)bh * a.n_split * PART;
    float m = -INFINITY, l = 0.f;
    float4_t o = {0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < a.n_split; s0 += BATCH) {
        float4_t st[BATCH], d[BATCH];
#pragma unroll
        for (int u = 0; u < BATCH; ++u) {
            const float* const p = parts + min(s0 + u, a.n_split - 1) * PART;
            st[u] = *reinterpret_cast<const float4_t*>(p + 32 * D + 4 * q);
            d[u] = *reinterpret_cast<const float4_t*>(p + (quad * 32 + q) * 4);
        }
        float top = m;
#pragma unroll
        for (int u = 0; u < BATCH; ++u) top = fmaxf(top, st[u][0]);      // (past the last share: its own again)
        const float wa = top > -INFINITY ? fast_exp2(m - top) : 1.f;
        l *= wa; o *= wa; m = top;
#pragma unroll
        for (int u = 0; u < BATCH; ++u) {
            if (s0 + u < a.n_split) {
                // (-inf: a share that saw no key of this query, whose sums are zero, or nothing but NaN scores, whose sums are that)
                const float w = st[u][0] > -INFINITY ? fast_exp2(st[u][0] - top) : 0.f;
                l = __builtin_fmaf(st[u][1], w, l);
                o += d[u] * w;
            }
        }
    }
    const int b = bh / a.Hq, head = bh - b * a.Hq;
    const float inv = 1.0f / l;
    half_t* const orow = a.o + b * a.ob + head * a.oh + (int64_t)q * a.os;
    *reinterpret_cast<half4_t*>(orow + 4 * quad) = half4_t{(half_t)(o[0] * inv), (half_t)(o[1] * inv), (half_t)(o[2] * inv), (half_t)(o[3] * inv)};
    if (quad == 0 && a.lse) a.lse[(int64_t)bh * a.Sq + q] = (m + fast_log2(l)) * kLn2;
}
static hipError_t launch_share_pair(AttnArgs a, int64_t at, int head_dim, hipStream_t s) {      // at: byte of the workspace from which on the shares' results lie
    a.n_qtiles = 1; a.partial = 2; a.ws += at / 4;
    const dim3 g((unsigned)(a.B * a.Hq * a.n_split)), t(DNW * 64), m((unsigned)(a.B * a.Hq * head_dim / 32));
    if (head_dim == 128) hipLaunchKernelGGL((attn_decode_kernel<128, 1, 7>), g, t, 0, s, a); else hipLaunchKernelGGL((attn_decode_kernel<64, 1, 7>), g, t, 0, s, a);
    if (const hipError_t e = hipGetLastError(); e != hipSuccess) return e;
    if (head_dim == 128) hipLaunchKernelGGL(attn_decode_merge_kernel<128>, m, dim3(256), 0, s, a); else hipLaunchKernelGGL(attn_decode_merge_kernel<64>, m, dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_attn_decode(AttnArgs a, int head_dim, void* workspace, int64_t workspace_bytes, hipStream_t stream) {
    a.n_split = 1; a.ws = nullptr; a.partial = 0;
    const int64_t counters = counter_bytes((int64_t)a.B * a.Hq);
    if (workspace && a.Sq <= 32 && !a.col_sum && !a.col_sumsq && !a.probs && !a.k_norm) {
        const int64_t own = attn_decode_workspace_bytes(a.B, a.Hq, a.Sq, a.Skv, head_dim);
        const int64_t need = own > 0 ? own : a.noise ? 0 : attn_few_query_workspace_bytes(a.B, a.Hq, a.Hkv, a.Sq, a.Skv, head_dim);
        if (need > 0 && workspace_bytes >= need) {
            a.ws = static_cast<float*>(workspace);
            if (!a.noise) {
                a.n_split = few_query_shares(a.B * a.Hq, a.B * a.Hkv, a.Skv, head_dim);
                if (a.n_split > 1) return launch_share_pair(a, own > 0 ? counters : kCounterRoom, head_dim, stream);
            } else a.n_split = decode_splits(a.B * a.Hq, a.Skv);
        }
    }
    const int stat_shares = workspace && (a.col_sum || a.col_sumsq) && !a.probs && !a.k_norm ?
        attn_decode_stat_shares(a.B, a.Hq, a.Hkv, a.Sq, a.Skv, head_dim, a.noise != nullptr, workspace_bytes) : 0;
    if (a.mean_std && stat_shares == 0) return hipErrorInvalidValue;      // (the single launch has the sums only)
    if (stat_shares > 0) {
        a.n_split = stat_shares; a.ws = static_cast<float*>(workspace) + counters / 4; a.partial = 1; a.n_qtiles = 1;
        const dim3 g((unsigned)(a.B * a.Hq * stat_shares)), t(DNW * 64);
        const int nz = !a.noise ? 0 : a.n16 ? 2 : 1;
#define TRN_DEC_PAIR(D_, N_) do { hipLaunchKernelGGL((attn_decode_kernel<D_, 1, N_ ? N_ : 7>), g, t, 0, stream, a); hipLaunchKernelGGL((attn_decode_kernel<D_, 1, N_ + 8>), g, t, 0, stream, a); } while (0)
        if (head_dim == 128) { if (nz == 0) TRN_DEC_PAIR(128, 0); else if (nz == 1) TRN_DEC_PAIR(128, 1); else TRN_DEC_PAIR(128, 2); }
        else { if (nz == 0) TRN_DEC_PAIR(64, 0); else if (nz == 1) TRN_DEC_PAIR(64, 1); else TRN_DEC_PAIR(64, 2); }
#undef TRN_DEC_PAIR
        return hipGetLastError();
    }
    // Without a key split: share V's columns out over workgroups while that still leaves every workgroup 32 columns
    // and the grid within one workgroup per CU (32 heads of 128: 4 shares; 71 heads of 64: 2).  Few queries on a short
    // cache are left alone: below some 8 blocks per wave-round the fixed part of a launch is all there is.
    a.n_qtiles = (a.Sq + 31) / 32;
    const int64_t n_bh = (int64_t)a.B * a.Hq;
    const int ds = a.n_split == 1 ? decode_col_shares(n_bh * a.n_qtiles, a.Sq, a.Skv, head_dim) : 1;
    const int64_t heads8 = (n_bh + 7) / 8;
    a.spread = decode_spread(n_bh, a.n_qtiles, ds) ? 1 : 0;
    const int64_t grid = a.spread ? (n_bh * a.n_qtiles + 7) / 8 * 8 * ds : ds > 1 || a.n_qtiles > 1 ? heads8 * 8 * ds * a.n_qtiles : n_bh * a.n_split;
    if (grid > 0x7fffffffLL) return hipErrorInvalidValue;
    const dim3 g((unsigned)grid), t(DNW * 64);
#define TRN_DEC(D_, DS_, N_) hipLaunchKernelGGL((attn_decode_kernel<D_, DS_, N_>), g, t, 0, stream, a)
    // (as the kernel deals them out: blocks of 32 keys to the eight waves in turn; the un-reduced probabilities come from the sweep)
    const bool keep = decode_keeps(a.B, a.Hq, a.Sq, a.Skv, head_dim, a.noise != nullptr) && a.n_split == 1 && (a.col_sum || a.col_sumsq) && !a.probs;
#define TRN_DEC_NZ(D_, DS_) do { if (keep) { if (!a.noise) TRN_DEC(D_, DS_, 4); else if (a.n16) TRN_DEC(D_, DS_, 6); else TRN_DEC(D_, DS_, 5); } else if (a.k_norm) TRN_DEC(D_, DS_, 3); else if (!a.noise) TRN_DEC(D_, DS_, 0); else if (a.n16) TRN_DEC(D_, DS_, 2); else TRN_DEC(D_, DS_, 1); } while (0)
    if (head_dim == 128) { if (ds == 4) TRN_DEC_NZ(128, 4); else if (ds == 2) TRN_DEC_NZ(128, 2); else TRN_DEC_NZ(128, 1); }
    else { if (ds == 2) TRN_DEC_NZ(64, 2); else TRN_DEC_NZ(64, 1); }
#undef TRN_DEC_NZ
#undef TRN_DEC
    return hipGetLastError();
}

}  // namespace trn

// ---- the entry point that allocates nothing ------------------------------------------------------------------------
// The split-key path needs device memory beyond its inputs and outputs (arrival counters and the shares' partial
// results).  For callers that cannot allocate, that memory is a file-scope device array: every GPU the library runs
// on holds its own copy of it, at its own address, until the process ends.  On the host the array's NAME is only a
// handle for hipGetSymbolAddress; the address that kernels, fills and copies take is the one that call returns for
// the device that is current, looked up once per device and kept.
static __device__ __align__(256) unsigned char scratch[TRN_ATTN_NOALLOC_SCRATCH_BYTES];

namespace trn {

constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mutex;
static void* g_scratch_ptr[kMaxDevices];      // device address of `scratch` on each device, null until looked up

// Device address of the scratch array on the current device (looked up on first use; nothing is allocated: the
// array is part of the code object).  Returns nullptr if the runtime refuses.
void* attn_static_scratch() {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return nullptr;
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess) return nullptr;
        g_scratch_ptr[dev] = p;
    }
    return g_scratch_ptr[dev];
}

// Zeroes n dwords (a kernel rather than a memset node, so that the call can be recorded into a graph).
__global__ __launch_bounds__(256) void fill_zero_kernel(unsigned* p, int n) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) p[i] = 0u;
}

}  // namespace trn

extern "C" int trn_attn_fwd_noalloc_f16(const trn_attn_desc* d, const void* q, const void* k, const void* v, void* o,
                                        float* lse, const void* gamma_q, const float* noise, float* lse_pert,
                                        void* stream) {
    using namespace trn;
    if (!d) return TRN_E_NULL;
    const int64_t need = trn_attn_workspace_bytes(d);
    if (need == 0)      // a shape whose kernels use no scratch memory (or an invalid one: reported by the checks below)
        return attn_forward(d, q, k, v, o, lse, gamma_q, noise, lse_pert, nullptr, 0, nullptr, nullptr, stream);
    if (need > (int64_t)TRN_ATTN_NOALLOC_SCRATCH_BYTES) return TRN_E_SCRATCH;
    void* ws = attn_static_scratch();
    if (!ws) return TRN_E_LAUNCH;
    // The array keeps whatever the last call on this device left.  The shares are rewritten by every launch before
    // they are read; the arrival counters, of calls with noise, must start at zero, so they are cleared here (the kernel also
    // leaves them at zero, but a launch that failed half way would not have).
    if (noise) {
        const int n_counters = (int)(((int64_t)d->batch * d->n_q_heads + 63) / 64) * 64;
        hipLaunchKernelGGL(fill_zero_kernel, dim3((n_counters + 255) / 256), dim3(256), 0, (hipStream_t)stream,
                           static_cast<unsigned*>(ws), n_counters);
        if (hipGetLastError() != hipSuccess) return TRN_E_LAUNCH;
    }
    return attn_forward(d, q, k, v, o, lse, gamma_q, noise, lse_pert, ws, TRN_ATTN_NOALLOC_SCRATCH_BYTES, nullptr, nullptr, stream);
}
