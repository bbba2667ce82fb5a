// Flash attention forward for gfx950 on the 32x32x16 MFMA: O = softmax(scale * Q K^T [+causal]) V, GQA/MQA,
// head_dim 64/128.  This file holds the entry points, and the kernel that runs when the scores are perturbed
// (KeyFormer: one lane owns a whole query row here, which is what the noise stream wants); plain attention runs
// on the 16x16x32 kernel of attn_fwd16.hip.
//
// Formulation.  Everything is computed TRANSPOSED so that a lane owns one query:
//     S^T[key][query] = K[key][:] . Q[query][:]     (MFMA 32x32x16: A = K tile from LDS, B = Q^T in registers)
//     O^T[d][query]  += V^T[d][key] * P^T[key][query]   (A = V^T tile from LDS, B = P^T straight from the
//                                                         S^T accumulator registers, rounded to fp16)
// In the 32x32 accumulator layout lane l holds column l%32 (the query) and 16 of the 32 rows (keys), so the
// softmax row max / row sum are in-lane reductions plus ONE exchange with lane l^32, the running max and
// normaliser are one scalar per lane, the O rescale needs no shuffles, and P never touches LDS: the MFMA
// contraction index may be permuted freely, so the accumulator's key order is matched by the order in
// which V^T is fetched.
//
// Workgroup: 256 threads = 4 waves, 128 queries (32 per wave); K/V tiles of BN keys go straight from global
// memory into double-buffered LDS (buffer_load ... lds, no register staging), row-major with an XOR chunk
// swizzle; the V^T A-operand is fetched with the gfx950 transposing LDS read ds_read_b64_tr_b16, so V needs
// no transposition in memory or on the way in.
// Grid: one workgroup per (query tile, batch, head), heaviest (latest) query tiles first; consecutive
// workgroup ids map to different KV heads so that the query heads sharing a KV head land on the same XCD
// (ids are dealt round-robin to the 8 XCDs) and hit its L2.
#include "attn.h"
#include <type_traits>

namespace trn {

#if defined(__HIP_DEVICE_COMPILE__)   // buffer-descriptor types and LDS-load builtins exist in the device pass only;
                                      // the host pass needs just the launch stubs
// N16: fp16 noise (fp32 otherwise).  NT: the noise is requested with the non-temporal hint.  SPLIT: the eight waves are two
// groups of four on the same 128 queries, each taking every other 64-key tile through stages of its own; their results are
// merged through LDS at the end.
template <int D, int NW, bool N16, bool NT, bool SPLIT>
__device__ __forceinline__ void attn_fwd_body(const AttnArgs& a) {
    static_assert(!SPLIT || NW == 8, "two groups of four waves");
    constexpr int GW = SPLIT ? 4 : NW;       // waves that share the K / V stages
    constexpr int NG = SPLIT ? 2 : 1;        // groups with stages of their own
    constexpr int KSTEP = SPLIT ? 128 : 64;  // keys from one tile of a wave to its next
    constexpr int BN = 64;       // keys per LDS stage (two 32-key blocks)
    constexpr int NS = D / 16;   // MFMA slots per phase: k-steps of S^T = K Q^T, and (2 key halves) x (D/32) of P V
    constexpr int NDB = D / 32;  // 32-wide blocks of head_dim in O^T
    constexpr int EPI = 16 / NS; // score elements converted per slot
    constexpr int CPR = D / 8;   // 16-byte chunks per row
    constexpr int RPI = 64 / CPR;            // stage rows covered by one wave-wide 1 KB load
    constexpr int NI = BN / (RPI * GW);      // such loads per wave per stage (K and V each)
    constexpr int BM = 32 * GW;              // queries per workgroup, 32 a wave
    // Two stages each for K and V, as FOUR separate arrays: the compiler orders an LDS read after every
    // outstanding global->LDS load that may alias it, and only distinct variables are provably disjoint --
    // with one [2][..] array every LDS read would wait for the prefetch that was just issued.
    __shared__ __attribute__((aligned(1024))) half_t Ks0_[NG * BN * D];
    __shared__ __attribute__((aligned(1024))) half_t Ks1_[NG * BN * D];
    __shared__ __attribute__((aligned(1024))) half_t Vs0_[NG * BN * D];
    __shared__ __attribute__((aligned(1024))) half_t Vs1_[NG * BN * D];
    // the waves' noise blocks on their way from whole row pieces, as they are fetched, to the accumulator layout
    constexpr int NSZ = N16 ? 2 : 4;
    __shared__ __attribute__((aligned(1024))) char Nt[NW * 1024 * NSZ];

    const int tid = threadIdx.x, lane = tid & 63, c = lane & 31, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int grp = SPLIT ? wave >> 2 : 0, gw = SPLIT ? wave & 3 : wave;
    half_t* const Ks0 = Ks0_ + grp * BN * D;
    half_t* const Ks1 = Ks1_ + grp * BN * D;
    half_t* const Vs0 = Vs0_ + grp * BN * D;
    half_t* const Vs1 = Vs1_ + grp * BN * D;
    const int kfirst = grp * BN;                        // first key of this wave's first tile

    // ---- which (query tile, batch, head): heavy tiles first, KV heads interleaved across ids
    const int tile_no = a.heads.all.of(blockIdx.x), qt = a.n_qtiles - 1 - tile_no;
    int b, kvh, g;
    a.heads.find(blockIdx.x - tile_no * a.heads.all.d, b, kvh, g);
    const int head = kvh * a.heads.G + g;

    const int off = a.Skv - a.Sq;                       // causal: query i sees keys <= i + off
    const int q0 = qt * BM;
    const int wq0 = q0 + gw * 32;                       // first query of this wave
    const int qrow = wq0 + c;                           // this lane's query
    const int qrow_ld = qrow < a.Sq ? qrow : a.Sq - 1;  // clamp loads; stores are predicated

    // ---- Q^T B-operands: lane holds Q[qrow][ks*16 + 8h .. +7]
    half8_t qB[NS];
    {
        const half_t* qp = a.q + b * a.qb + head * a.qh + (int64_t)qrow_ld * a.qs + 8 * h;
#pragma unroll
        for (int ks = 0; ks < NS; ++ks) qB[ks] = *reinterpret_cast<const half8_t*>(qp + ks * 16);
        if (a.q_norm) {   // fused per-head RMSNorm of the query row (other half of the row is in lane^32)
            float ss = 0.f;
#pragma unroll
            for (int ks = 0; ks < NS; ++ks)
#pragma unroll
                for (int e = 0; e < 8; ++e) { float f = (float)qB[ks][e]; ss += f * f; }
            ss = half_sum(ss);
            const float rstd = 1.0f / __builtin_sqrtf(ss / (float)D + a.q_eps);
#pragma unroll
            for (int ks = 0; ks < NS; ++ks) {
                half8_t gq;
                if (a.gamma_q) gq = *reinterpret_cast<const half8_t*>(a.gamma_q + ks * 16 + 8 * h);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    float y = (float)qB[ks][e] * rstd;
                    if (a.gamma_q) y = (float)gq[e] * y;
                    qB[ks][e] = (half_t)y;
                }
            }
        }
    }

    // ---- LDS read offsets (halfs), lane constants.  K operand: row c of a 32-key block, logical chunk 2ks+h.
    int koff[NS];
#pragma unroll
    for (int ks = 0; ks < NS; ++ks) koff[ks] = c * D + (((2 * ks + h) ^ swz<D>(c)) << 3);
    // V^T operand through the transposing read: in each 16-lane group lanes 4r..4r+3 supply stage row r
    // (4 consecutive 8-byte pieces); this lane's piece is row 4h + (lane%16)/4 [+8], head_dim columns
    // db*32 + 16*((lane/16)%2) + 4*(lane%4).
    int voff_lo[NDB], voff_hi[NDB];
    {
        const int rl = 4 * h + ((lane & 15) >> 2), rh = rl + 8;
        const int lc = 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1), sub = (lane & 1) * 4;
#pragma unroll
        for (int db = 0; db < NDB; ++db) {
            voff_lo[db] = rl * D + (((db * 4 + lc) ^ swz<D>(rl)) << 3) + sub;
            voff_hi[db] = rh * D + (((db * 4 + lc) ^ swz<D>(rh)) << 3) + sub;
        }
    }

    float16_t oacc[NDB];
#pragma unroll
    for (int i = 0; i < NDB; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[i][r] = 0.f;
    float m = -INFINITY, l = 0.f;      // reference max (log2 domain) and this lane's partial row sum
    float m2 = 0.f, l2 = 0.f;          // same for the perturbed scores: reference (finite; meaningful once have2) and sum
    bool have2 = false;

    int ntiles = (a.Skv + BN - 1) / BN;
    if (a.causal) ntiles = min(ntiles, (min(q0 + BM - 1, a.Sq - 1) + off) / BN + 1);

    // KeyFormer noise, the HBM stream that bounds this kernel: a 32 x 32 block per wave and step, requested two steps before it
    // is used (buffer loads: keys or rows past the end read as zeros or as another row's and are masked anyway).  A load
    // takes whole row pieces, eight lanes a row of 32 keys; in the accumulator layout, a row per lane, it touches 32 lines and
    // a CU serves such loads at 16 bytes a clock instead of 64 -- more than the arithmetic of a step takes, and every wave
    // waits to issue behind them (71 heads of 64, 2752 keys, fp16: 221 -> 186 us; 32 of 128, 2048, fp32: 124 -> 109, streamed
    // past the caches 98).  On arrival the block goes through a wave-private part of LDS into the accumulator layout
    // (LDS operations of one wave execute in order: no barrier).  fp16 noise: three dwords around 4 keys, shifted on arrival.
    typedef typename std::conditional<N16, uint3_t, float4_t>::type noise_t;
    typedef typename std::conditional<N16, half4_t, float4_t>::type nquad_t;
    const void* nbase = reinterpret_cast<const char*>(a.noise) + (b * a.nb + head * a.nh) * NSZ;
    const HalfNoise hn(nbase, N16 ? a.Sq : 1, N16 ? a.ns : 0, N16 ? a.Skv : 0);
    const __amdgpu_buffer_rsrc_t nrs = N16 ? hn.rs : __builtin_amdgcn_make_buffer_rsrc(
        (void*)nbase, 0, (int)(((int64_t)(a.Sq - 1) * a.ns + a.Skv) * 4), 0x00020000);
    int nsh = 0, nrow[4];              // byte offsets of the wave's rows 0, 8, 16, 24: at most 7 rows past the last are asked for
    const int64_t nfirst = (lane >> 3) * a.ns + 4 * (lane & 7);
#pragma unroll
    for (int i = 0; i < 4; ++i) nrow[i] = (int)(min(wq0 + 8 * i, (a.Sq - 1) & ~7) * a.ns * NSZ);      // (a multiple of 8 rows: dwords)
    const int nvo = N16 ? hn.row(nfirst, nsh) : (int)(nfirst * 4);
    noise_t gpre0[4], gpre1[4];        // even / odd 32-key blocks: each refilled two blocks ahead, as soon as it is used
    auto fetch_noise = [&](int key0, noise_t (&gpre)[4]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if constexpr (N16) gpre[i] = __builtin_bit_cast(noise_t, __builtin_amdgcn_raw_buffer_load_b96(nrs, nvo, nrow[i] + key0 * 2, NT ? 2 : 0));
            else gpre[i] = __builtin_bit_cast(noise_t, __builtin_amdgcn_raw_buffer_load_b128(nrs, nvo, nrow[i] + key0 * 4, NT ? 2 : 0));
        }
    };
    // 4 keys of row r at place q ^ (r/2) % 8 of the row's eight (fp16, two rows more to a line of the 64 banks: q ^ (r/4) % 8),
    // written as fetched, read as row c, quads 2i + h: both conflict-free
    nquad_t* const nt = reinterpret_cast<nquad_t*>(Nt + wave * 1024 * NSZ);
    int nt_wr[2], nt_rd[4];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int r = 8 * i + (lane >> 3);
        nt_wr[i] = r * 8 + ((lane & 7) ^ ((r >> (N16 ? 2 : 1)) & 7));
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) nt_rd[i] = c * 8 + ((2 * i + h) ^ ((c >> (N16 ? 2 : 1)) & 7));
    auto stash_noise = [&](const noise_t (&gpre)[4]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            // (the place of rows 16 further differs in bit 2 where the swizzle counts pairs of rows or fours of them)
            const int at = N16 ? (i < 2 ? nt_wr[i] : (nt_wr[i & 1] ^ 4) + 128) : nt_wr[i & 1] + (i >> 1) * 128;
            if constexpr (N16) nt[at] = half_noise4(gpre[i], nsh); else nt[at] = gpre[i];
        }
    };
    auto noise_quads = [&](nquad_t (&g)[4]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) g[i] = nt[nt_rd[i]];
    };

    // ---- staging: direct global -> LDS loads.  Buffer descriptors give zero fill for keys past the end
    // (an all-zero V row times P = 0 contributes nothing; garbage could be NaN).
    const __amdgpu_buffer_rsrc_t krs = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(a.k + b * a.kb + kvh * a.kh), 0, (int)(((int64_t)(a.Skv - 1) * a.ks + D) * 2), 0x00020000);
    const __amdgpu_buffer_rsrc_t vrs = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(a.v + b * a.vb + kvh * a.vh), 0, (int)(((int64_t)(a.Skv - 1) * a.vs + D) * 2), 0x00020000);
    const int st_row = gw * RPI + lane / CPR;                      // this lane's row within each 4*RPI-row group
    const int st_chunk = (lane % CPR) ^ swz<D>(st_row);             // LDS slot lane%CPR of that row holds this logical chunk
    const int kvo = (int)(st_row * a.ks * 2) + st_chunk * 16;       // per-lane byte offsets within a stage
    const int vvo = (int)(st_row * a.vs * 2) + st_chunk * 16;
    const int krow_bytes = (int)(RPI * a.ks * 2), vrow_bytes = (int)(RPI * a.vs * 2);
    const int ktile_bytes = (int)(KSTEP * a.ks * 2), vtile_bytes = (int)(KSTEP * a.vs * 2);
    const int kgrp_bytes = (int)(kfirst * a.ks * 2), vgrp_bytes = (int)(kfirst * a.vs * 2);
#define TRN_FETCH_K(jt_, dst_) fetch_tile<NI, D, GW>(krs, &dst_[gw * RPI * D], kvo, kgrp_bytes + (jt_) * ktile_bytes, krow_bytes)
#define TRN_FETCH_V(jt_, dst_) fetch_tile<NI, D, GW>(vrs, &dst_[gw * RPI * D], vvo, vgrp_bytes + (jt_) * vtile_bytes, vrow_bytes)

    const float16_t zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    const int last_key = min(a.Skv - 1, a.causal ? qrow + off : a.Skv - 1);    // the last key this lane's query sees

    // Scores of a 32-key block starting at key0, just produced: (KeyFormer) fold them into the perturbed
    // row normaliser; mask; block max against the LAZY reference max m.  m is only raised when some row's
    // true running max exceeds it by more than 2^8: probabilities are then at most 256 (exact in fp16's
    // range, fp32 sums), O and l stay relative to the same m so the final O/l and m + log2(l) are unchanged,
    // and the 16*NDB-multiply rescale of O^T runs on the first block or two only instead of on most blocks.
    // Returns whether a rescale is due (wave-uniform) and the candidate max.
    // (The form for blocks that may need the mask; the steps of the plain loop do the same between their MFMAs.)
    auto reduce_block = [&](float16_t& sx, int key0, float& smax, const nquad_t (&g)[4], noise_t (&gpre)[4]) __attribute__((always_inline)) {
        const int last = last_key - key0 - 4 * h;      // as an offset from the lane's first key
        // Row normaliser of the perturbed scores z = s*c2 + g*c3 (log2 domain), with a lazy reference like the
        // main softmax: d = z - m2 comes straight out of two fused multiply-adds, and m2 is only raised when some d
        // exceeds 8 (the sum lives in fp32: 2^8 of head-room is harmless) or nothing has been summed yet.
        const float nref = -m2;
        float16_t d;
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float dd = __builtin_fmaf(sx[r4 * 4 + e], a.c2, __builtin_fmaf((float)g[r4][e], a.c3, nref));
                d[r4 * 4 + e] = 8 * r4 + e <= last ? dd : -INFINITY;
            }
        }
        fetch_noise(key0 + KSTEP, gpre); // the next block of the same parity, two pipeline steps ahead of its use
        // The test runs on the lane's own 16 keys; the exchange with the other lane of the query (m2 and have2 are
        // shared by the pair) is made on the rare path only -- if either lane of a pair wants the raise, the
        // wave-wide vote takes every lane there.
        const float down = max16_bare(d);
        if (__builtin_amdgcn_ballot_w64(down > 8.0f || (!have2 && down > -INFINITY)) != 0) {     // rare after a row's first block
            const float dmax = half_max(down);
            const bool seen = dmax > -INFINITY;            // a block can be entirely masked for this row pair
            const bool raise = dmax > 8.0f || (!have2 && seen);
            const float shift = raise ? dmax : 0.f;
            l2 = have2 ? l2 * fast_exp2(-shift) : 0.f;     // (a first reference below -128 would make the power infinite)
            m2 += shift;
#pragma unroll
            for (int r = 0; r < 16; ++r) d[r] -= shift;
            have2 = have2 || seen;
        }
        float sum = 0.f;
#pragma unroll
        for (int r = 0; r < 16; ++r) sum += fast_exp2(d[r]);
        l2 += sum;
#pragma unroll
        for (int r = 0; r < 16; ++r)
            sx[r] = 8 * (r / 4) + (r % 4) <= last ? sx[r] : -INFINITY;      // (a select: stale-LDS garbage past the last block never propagates)
        smax = max16_bare(sx) * a.c1;          // over the lane's own keys; the pair's maximum is formed in rescale()
        return __builtin_amdgcn_ballot_w64(smax > m + 8.0f) != 0;
    };
    auto rescale = [&](float smax_own) __attribute__((always_inline)) {
        const float smax = half_max(smax_own);
        const float mnew = fmaxf(m, smax);
        const float alpha = fast_exp2(m - mnew);
        l *= alpha;
#pragma unroll
        for (int i = 0; i < NDB; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) oacc[i][r] *= alpha;
        m = mnew;
    };

    constexpr int NQ = 2;   // operand look-ahead in MFMA slots (deeper windows measured the same)
    half8_t ka[NQ];    // K operands of the next block's S^T: a rolling window NQ MFMA slots ahead of use
    half8_t va[NQ];    // V^T operands of this block's P V: likewise

    // One pipeline step for block B whose scores sc are complete, masked and reflected in m:
    //   phase A: MFMA: S^T of block B+1                  | VALU: P = exp2(sc*c1 - m), fp16, row sum
    //   phase B: MFMA: O^T += V^T P^T                    | VALU: mask + max of block B+1's scores
    // A wave issues in order and an MFMA holds the matrix pipe for 8 passes, so program order IS the
    // schedule: one MFMA, its share of the VALU work and one LDS operand request per slot, with
    // sched_barrier to keep the compiler from regrouping.  Each operand is requested NQ slots before its
    // MFMA, into the register its predecessor just vacated:
    //   phase A slot i < NS-NQ : K operand i+NQ of block B+1 (K1)   later slots : V^T operand i+NQ-NS of block B
    //   phase B slot i < NS-NQ : V^T operand i+NQ of block B        later slots : K operand i+NQ-NS of block B+2 (K2)
    // With SYNC (first block of a 64-key tile) the tile hand-over sits NQ slots before the end of phase A: by
    // then every wave has made its last read of the tile's own K stage (block B+1's last operands) and of the
    // previous tile's V stage, so after the barrier those two stages are refilled (K two tiles ahead, V one
    // tile ahead) and all later LDS reads of this and the next step go to the stages that just became visible.
    auto step = [&](auto plain_tag, auto sync_tag, float16_t& sc, float16_t& sn, const half_t* Vblk, const half_t* K1,
                    const half_t* K2, int key0_next, auto&& handover, auto&& refill, noise_t (&gpre)[4]) __attribute__((always_inline)) {
        constexpr bool SYNC = decltype(sync_tag)::value, PLAIN = decltype(plain_tag)::value;
        // The row sum is taken over the fp16-rounded P (v_dot2_f32_f16 against ones, fp32 accumulate),
        // i.e. over exactly the values that multiply V.
        const half2_t ones = {(half_t)1.f, (half_t)1.f};
        half8_t pB[2];
        auto load_v = [&](int op, int reg) __attribute__((always_inline)) {
            const half_t* vp = Vblk + 16 * (op / NDB) * D;
            half4_t lo = lds_read_tr16(vp + voff_lo[op % NDB]);   // keys +0..3 of this lane half, dim db*32+c
            half4_t hi = lds_read_tr16(vp + voff_hi[op % NDB]);   // keys +8..11
            va[reg] = half8_t{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        };
        nquad_t g[4];
        // ---- phase A ----
#pragma unroll
        for (int i = 0; i < NS; ++i) {
            if constexpr (SYNC) {
                if (i == NS - NQ) handover();
            }
            if (i == NS - 2) stash_noise(gpre);
            if (i == NS - 1) noise_quads(g);
            sn = mfma32(ka[i % NQ], qB[i], i == 0 ? zero : sn);
            if (i + NQ < NS) ka[i % NQ] = *reinterpret_cast<const half8_t*>(&K1[koff[i + NQ]]);
            else load_v(i + NQ - NS, i % NQ);
#pragma unroll
            for (int e = 0; e < EPI; e += 2) {
                const int r = i * EPI + e;
                const float p0 = fast_exp2(__builtin_fmaf(sc[r], a.c1, -m));
                const float p1 = fast_exp2(__builtin_fmaf(sc[r + 1], a.c1, -m));
                const half2_t pp = {(half_t)p0, (half_t)p1};
                l = __builtin_amdgcn_fdot2(pp, ones, l, false);
                pB[r / 8][r % 8] = pp[0]; pB[r / 8][r % 8 + 1] = pp[1];
            }
            asm volatile("" : "+v"(l));
            __builtin_amdgcn_sched_barrier(0);
        }
        // ---- phase B ----
        float smax = 0.f;
        bool due = false;
        // No mask: the perturbed scores are exponentiated and summed between the MFMAs, two scores at a time, against the
        // reference as it stands.  That it has to be raised shows in the sum of the lane's 16 (over 256: some score lies more
        // than 4 above it; none more than 8 otherwise), and the block's sum is then formed again (rare after a row's first).
        const float nref = -m2;
        float top = -INFINITY, sum = 0.f;
        auto perturbed = [&](int r, float ref) __attribute__((always_inline)) {
            return __builtin_fmaf(sn[r], a.c2, __builtin_fmaf((float)g[r / 4][r % 4], a.c3, ref));
        };
#pragma unroll
        for (int i = 0; i < NS; ++i) {
            oacc[i % NDB] = mfma32(va[i % NQ], pB[i / NDB], oacc[i % NDB]);
            if (i + NQ < NS) load_v(i + NQ, i % NQ);
            else ka[i % NQ] = *reinterpret_cast<const half8_t*>(&K2[koff[i + NQ - NS]]);
            if constexpr (SYNC) {
                if (i < NS / 2) {
#pragma unroll
                    for (int k = 0; k < 4 * NI / NS; ++k) refill(i * (4 * NI / NS) + k);
                }
            }
            if constexpr (PLAIN) {
                // scores [first(i), first(i + 1)) in slot i: none in slot 0, whose MFMA covers the end of the score chain
                auto first = [](int k) { return NS == 8 ? (k == 8 ? 16 : k < 1 ? 0 : 2 * (k - 1)) : k == 4 ? 16 : k < 2 ? 0 : k == 2 ? 4 : 10; };
#pragma unroll
                for (int r = first(i); r < first(i + 1); r += 2) {
                    const float d0 = perturbed(r, nref), d1 = perturbed(r + 1, nref);
                    top = max3_after(top, sn[r], sn[r + 1], d1);
                    sum += fast_exp2(d0);
                    sum += fast_exp2(d1);
                    asm volatile("" : "+v"(sum));     // (left alone the compiler moves all of this behind the last MFMA)
                }
            } else if (i == NS / 2) due = reduce_block(sn, key0_next, smax, g, gpre);
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (PLAIN) {
            smax = top * a.c1;
            if (__builtin_amdgcn_ballot_w64(!have2 || sum > 256.0f || smax > m + 8.0f) != 0) {
                float down = -INFINITY;
#pragma unroll
                for (int r = 0; r < 16; ++r) down = fmaxf(down, perturbed(r, nref));
                const float dmax = half_max(down);
                const bool seen = dmax > -INFINITY, raise = dmax > 4.0f || (!have2 && seen);
                const float shift = raise ? dmax : 0.f;
                l2 = have2 ? l2 * fast_exp2(-shift) : 0.f;     // (as in reduce_block)
                m2 += shift;
                have2 = have2 || seen;
                sum = 0.f;
#pragma unroll
                for (int r = 0; r < 16; ++r) sum += fast_exp2(perturbed(r, nref) - shift);
                due = __builtin_amdgcn_ballot_w64(smax > m + 8.0f) != 0;
            }
            l2 += sum;
            fetch_noise(key0_next + KSTEP, gpre);
        }
        if (due) rescale(smax);
    };

    // ---- prologue: K stages 0 and 1 and V stage 0; scores of block 0; first K operands of block 1 ----
    // In the order in which they are waited for, so that the start does not wait for all: the first tile's hand-over, for instance, waits
    // for V and the second K with the eight noise requests behind them still under way.  Whole calls, us, all waited for / so: 8 x 32 heads of
    // 128, 180 keys, fp16 23.0 / 22.4, 71 of 64, 250 19.1 / 18.75, 32 of 128, 1501 69.1 / 68.8, 4096 fp32 the same.
    TRN_FETCH_K(0, Ks0);
    __builtin_amdgcn_sched_barrier(0);
    fetch_noise(kfirst, gpre0);
    __builtin_amdgcn_sched_barrier(0);
    TRN_FETCH_V(0, Vs0);
    TRN_FETCH_K(1, Ks1);
    __builtin_amdgcn_sched_barrier(0);
    fetch_noise(kfirst + 32, gpre1);
    {
        constexpr int kBehind = 2 * NI + 8;
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(0x0f70 | (kBehind & 15) | ((kBehind >> 4) << 14));
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
    }

    float16_t sA, sB;                       // scores of the current / next 32-key block (ping-pong)
    {
        half8_t k0[NS];
#pragma unroll
        for (int i = 0; i < NS; ++i) k0[i] = *reinterpret_cast<const half8_t*>(&Ks0[koff[i]]);
#pragma unroll
        for (int i = 0; i < NS; ++i) sA = mfma32(k0[i], qB[i], i == 0 ? zero : sA);
#pragma unroll
        for (int i = 0; i < NQ; ++i) ka[i] = *reinterpret_cast<const half8_t*>(&Ks0[32 * D + koff[i]]);
        float smax;
        nquad_t g[4];
        stash_noise(gpre0);
        noise_quads(g);
        if (reduce_block(sA, kfirst, smax, g, gpre0)) rescale(smax);
    }

    // One 64-key tile jt.  Kc = its own K stage (block 1 still has operands to give), Kn = the next tile's
    // K stage, Vc = its V stage, Vn = the other V stage.
    auto tile = [&](auto plain_tag, int jt, half_t* Kc, const half_t* Kn, const half_t* Vc, half_t* Vn) __attribute__((always_inline)) {
        const int kv0 = kfirst + jt * KSTEP;
        auto handover = [&]() __attribute__((always_inline)) {
            // this wave's share of stages Kn and Vc is in LDS: everything but the noise requests of the two
            // steps since the stages were requested (2 x 4 loads, issued behind them) has returned
            __builtin_amdgcn_s_waitcnt(0x0f78);
            __syncthreads();                      // ... and everyone's; Kc and Vn have had their last readers
            // The refills are issued unconditionally (tiles past the end just fill stages
            // nobody reads): the compiler sizes its waits for the noise registers by the loads it KNOWS follow
            // them, and a conditional load counts as absent -- every noise use would drain the refills too.
        };
        auto refill = [&](int i) __attribute__((always_inline)) {
            if (i < NI) fetch_piece<D, GW>(vrs, &Vn[gw * RPI * D], vvo, vgrp_bytes + (jt + 1) * vtile_bytes, vrow_bytes, i);
            else fetch_piece<D, GW>(krs, &Kc[gw * RPI * D], kvo, kgrp_bytes + (jt + 2) * ktile_bytes, krow_bytes, i - NI);
        };
        auto none = [&]() __attribute__((always_inline)) {};
        auto none1 = [&](int) __attribute__((always_inline)) {};
        // (Past the last tile a K stage holds stale rows; scores computed from them are masked away.)
        step(plain_tag, std::true_type{}, sA, sB, Vc, Kc + 32 * D, Kn, kv0 + 32, handover, refill, gpre1);
        step(plain_tag, std::false_type{}, sB, sA, Vc + 32 * D, Kn, Kn + 32 * D, kv0 + KSTEP, none, none1, gpre0);
    };
    // Under a causal mask a wave computes the tiles that hold a key visible to one of its queries and for the rest only keeps
    // up the staging that it shares with the others.  The tiles whose successors need no mask have a loop of their own (whole
    // turns of the two stages), the tiles at the diagonal and at the end of the keys another.
    int nlive = ntiles;
    if (a.causal) nlive = min(ntiles, (min(wq0 + 31, a.Sq - 1) + off) / BN + 1);
    const int nloop = SPLIT ? (ntiles + 1) >> 1 : ntiles;
    if constexpr (SPLIT) nlive = (nlive - grp + 1) >> 1;
    if (wq0 >= a.Sq) nlive = 0;
    const int lim = (a.causal ? min(a.Skv, wq0 + off + 1) : a.Skv) - kfirst;     // keys that every query of the wave sees
    const int n_plain = min(nlive, lim >= KSTEP + 32 ? (lim - KSTEP - 32) / KSTEP + 1 : 0) & ~1;
    int jt = 0;
    for (; jt < n_plain; jt += 2) {
        tile(std::true_type{}, jt, Ks0, Ks1, Vs0, Vs1);
        tile(std::true_type{}, jt + 1, Ks1, Ks0, Vs1, Vs0);
    }
    for (; jt < nlive; jt += 2) {
        tile(std::false_type{}, jt, Ks0, Ks1, Vs0, Vs1);
        if (jt + 1 < nlive) tile(std::false_type{}, jt + 1, Ks1, Ks0, Vs1, Vs0);
    }
    for (jt = nlive; jt < nloop; ++jt) {
        half_t* Kc = (jt & 1) ? Ks1 : Ks0;
        half_t* Vn = (jt & 1) ? Vs0 : Vs1;
        __builtin_amdgcn_s_waitcnt(0x0f70);
        __syncthreads();
        if (jt + 2 < nloop) TRN_FETCH_K(jt + 2, Kc);
        if (jt + 1 < nloop) TRN_FETCH_V(jt + 1, Vn);
    }
#undef TRN_FETCH_K
#undef TRN_FETCH_V

    // ---- epilogue: normalise; transpose this wave's 32 x D tile through LDS so that the stores are whole
    // 16-byte-per-lane row segments (the accumulator layout would give 8-byte pieces scattered over 32 rows,
    // i.e. partial-line writes); LSEs ----
    __builtin_amdgcn_s_waitcnt(0x0f70);                // the refills past the last tile have landed ...
    __syncthreads();                                   // ... everywhere, and every wave is done with the K/V stages
    l = half_sum(l); l2 = half_sum(l2);
    if constexpr (SPLIT) {
        // The groups hold partial results of the same queries: waves w and w + 4 exchange the normalisers and halves of O^T
        // lane by lane, group 0 finishes the first D/2 columns, group 1 the others.  A query that saw no key of its group (or
        // none of finite perturbed score) has zero sums and weighs nothing.
        constexpr int NH = NDB / 2, kStat = D == 128 ? 5120 : 2560;      // (floats) behind the regions of the output's way through LDS
        if (!have2) m2 = -INFINITY;
        float4_t* stat = reinterpret_cast<float4_t*>(reinterpret_cast<float*>(Ks1_) + kStat);        // [8 waves][32 queries]
        if (h == 0) stat[wave * 32 + c] = float4_t{m, l, m2, l2};
        float4_t* mine = reinterpret_cast<float4_t*>(grp == 0 ? Ks0_ : Vs0_) + gw * NH * 256;
        const float4_t* theirs = reinterpret_cast<const float4_t*>(grp == 0 ? Vs0_ : Ks0_) + gw * NH * 256;
#pragma unroll
        for (int i = 0; i < NH; ++i)
#pragma unroll
            for (int r4 = 0; r4 < 4; ++r4) {
                const float16_t& o = grp == 0 ? oacc[NH + i] : oacc[i];
                mine[(i * 4 + r4) * 64 + lane] = float4_t{o[4 * r4], o[4 * r4 + 1], o[4 * r4 + 2], o[4 * r4 + 3]};
            }
        __syncthreads();
        const float4_t t = stat[(wave ^ 4) * 32 + c];
        const float ms = fmaxf(m, t[0]), m2s = fmaxf(m2, t[2]);
        const float wo = m == -INFINITY ? 0.f : fast_exp2(m - ms), wt = t[0] == -INFINITY ? 0.f : fast_exp2(t[0] - ms);
        l = l * wo + t[1] * wt; m = ms;
        l2 = (m2 == -INFINITY ? 0.f : l2 * fast_exp2(m2 - m2s)) + (t[2] == -INFINITY ? 0.f : t[3] * fast_exp2(t[2] - m2s));
        m2 = m2s == -INFINITY ? 0.f : m2s;
        const float inv = 1.0f / l;
        constexpr int DP = D / 2, OP = DP + 4, LPRW = DP / 8, RPS = 64 / LPRW;
        half_t* ot = (grp == 0 ? Vs1_ : Ks1_) + gw * 32 * OP;
        static_assert(4 * 32 * OP * 2 <= kStat * 4 && kStat * 4 + 4096 <= 2 * BN * D * 2, "the stage holds both");
#pragma unroll
        for (int i = 0; i < NH; ++i)
#pragma unroll
            for (int r4 = 0; r4 < 4; ++r4) {
                const float16_t& o = grp == 0 ? oacc[i] : oacc[NH + i];
                const float4_t u = theirs[(i * 4 + r4) * 64 + lane];
                half4_t ov;
#pragma unroll
                for (int e = 0; e < 4; ++e) ov[e] = (half_t)((o[4 * r4 + e] * wo + u[e] * wt) * inv);
                *reinterpret_cast<half4_t*>(&ot[c * OP + i * 32 + 8 * r4 + 4 * h]) = ov;
            }
        const int orow = lane / LPRW, ocol = (lane % LPRW) * 8;
        half_t* ob = a.o + b * a.ob + head * a.oh + grp * DP;
#pragma unroll
        for (int j = 0; j < 32 / RPS; ++j) {
            const int r = j * RPS + orow;
            const uint2_t lo = *reinterpret_cast<const uint2_t*>(&ot[r * OP + ocol]);
            const uint2_t hi = *reinterpret_cast<const uint2_t*>(&ot[r * OP + ocol + 4]);
            if (wq0 + r < a.Sq)
                store_out(ob + (int64_t)(wq0 + r) * a.os + ocol, uint4_t{lo.x, lo.y, hi.x, hi.y}, a.o_nt);
        }
        if (grp == 1) return;               // (the normalisers are written once)
    } else {
        // two passes of D/2 columns each, so that NW waves' staging regions fit in the four stage arrays
        const float inv = 1.0f / l;
        constexpr int DP = D / 2, OP = DP + 4;         // row pitch in halfs: 8-byte writes of 32 rows spread over all banks
        constexpr int LPRW = DP / 8, RPS = 64 / LPRW;  // lanes per output row segment, rows per store instruction
        static_assert(32 * OP * 2 <= BN * D * 2 / (NW / 4), "staging region too large");
        half_t* arr = (wave / (NW / 4)) == 0 ? Ks0 : (wave / (NW / 4)) == 1 ? Ks1 : (wave / (NW / 4)) == 2 ? Vs0 : Vs1;
        half_t* ot = arr + (wave % (NW / 4)) * (BN * D / (NW / 4));
        const int orow = lane / LPRW, ocol = (lane % LPRW) * 8;
        half_t* ob = a.o + b * a.ob + head * a.oh;
#pragma unroll
        for (int pass = 0; pass < 2; ++pass) {
#pragma unroll
            for (int dbl = 0; dbl < NDB / 2; ++dbl)
#pragma unroll
                for (int r4 = 0; r4 < 4; ++r4) {
                    half4_t ov;
#pragma unroll
                    for (int e = 0; e < 4; ++e) ov[e] = (half_t)(oacc[pass * (NDB / 2) + dbl][r4 * 4 + e] * inv);
                    *reinterpret_cast<half4_t*>(&ot[c * OP + dbl * 32 + 8 * r4 + 4 * h]) = ov;
                }
            // (LDS operations of one wave execute in order: no wait needed between its own writes and reads)
#pragma unroll
            for (int j = 0; j < 32 / RPS; ++j) {
                const int r = j * RPS + orow;
                const uint2_t lo = *reinterpret_cast<const uint2_t*>(&ot[r * OP + ocol]);
                const uint2_t hi = *reinterpret_cast<const uint2_t*>(&ot[r * OP + ocol + 4]);
                if (wq0 + r < a.Sq)
                    store_out(ob + (int64_t)(wq0 + r) * a.os + pass * DP + ocol, uint4_t{lo.x, lo.y, hi.x, hi.y}, a.o_nt);
            }
        }
    }
    if (qrow < a.Sq && h == 0 && a.lse) a.lse[((int64_t)b * a.Hq + head) * a.Sq + qrow] = (m + fast_log2(l)) * kLn2;
    if (qrow < a.Sq && h == 0) a.lse_pert[((int64_t)b * a.Hq + head) * a.Sq + qrow] = (m2 + fast_log2(l2)) * kLn2;
}
#endif

// Narrow: 4 waves, 128 queries, two workgroups per CU; Wide: 8 waves, 256 queries; Split: 8 waves on 128 queries, two groups
// that take every other key tile each.
enum class NoiseShape { Narrow, Wide, Split };

// fp32 noise.  USUAL: in the cache policy of the shape's usual sizes -- past the caches for 256 queries of 128, through them
// elsewhere -- or in the other one (see noise_streams()).
template <int D, int NW, bool USUAL>
__global__ __launch_bounds__(NW * 64, NW == 8 ? 1 : 2) void attn_fwd_kernel(const AttnArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
    attn_fwd_body<D, NW, false, (D == 128 && NW == 8) == USUAL, false>(a);
#endif
}
template <int D, int NW>
__global__ __launch_bounds__(NW * 64, NW == 8 ? 1 : 2) void attn_fwd_half_noise_kernel(const AttnArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
    attn_fwd_body<D, NW, true, false, false>(a);
#endif
}
template <int D, bool N16, bool NT>
__global__ __launch_bounds__(512, 1) void attn_fwd_split_kernel(const AttnArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
    attn_fwd_body<D, 8, N16, NT, true>(a);
#endif
}

template <int D, int NW>
static void launch_rows(const AttnArgs& a, bool stream_noise, const dim3& g, hipStream_t s) {
    const dim3 t(NW * 64);
    if (a.n16) hipLaunchKernelGGL((attn_fwd_half_noise_kernel<D, NW>), g, t, 0, s, a);
    else if (stream_noise == (D == 128 && NW == 8)) hipLaunchKernelGGL((attn_fwd_kernel<D, NW, true>), g, t, 0, s, a);
    else hipLaunchKernelGGL((attn_fwd_kernel<D, NW, false>), g, t, 0, s, a);
}

template <int D>
static hipError_t launch_fwd(AttnArgs a, NoiseShape shape, bool stream_noise, hipStream_t s) {
    const int rows = shape == NoiseShape::Wide ? 256 : 128;
    a.n_qtiles = (int)(((int64_t)a.Sq + rows - 1) / rows);
    const int64_t grid = (int64_t)a.n_qtiles * a.B * a.Hq;
    if (grid > 0x7fffffffLL) return hipErrorInvalidValue;
    const dim3 g((unsigned)grid);
    if (shape == NoiseShape::Wide) launch_rows<D, 8>(a, stream_noise, g, s);
    else if (shape == NoiseShape::Narrow) launch_rows<D, 4>(a, stream_noise, g, s);
    else if (a.n16) hipLaunchKernelGGL((attn_fwd_split_kernel<D, true, false>), g, dim3(512), 0, s, a);
    else if (stream_noise) hipLaunchKernelGGL((attn_fwd_split_kernel<D, false, true>), g, dim3(512), 0, s, a);
    else hipLaunchKernelGGL((attn_fwd_split_kernel<D, false, false>), g, dim3(512), 0, s, a);
    return hipGetLastError();
}

int validate_attn(const trn_attn_desc* d, bool need_v);
int validate_attn(const trn_attn_desc* d, bool need_v) {
    if (d->batch <= 0 || d->n_q_heads <= 0 || d->n_kv_heads <= 0 || d->seq_q <= 0 || d->seq_kv <= 0) return TRN_E_SHAPE;
    if (d->n_q_heads % d->n_kv_heads != 0) return TRN_E_SHAPE;
    if (d->head_dim != 64 && d->head_dim != 128) return TRN_E_UNSUPPORTED;
    if (d->causal && d->seq_kv < d->seq_q) return TRN_E_SHAPE;
    if (!(d->scale > 0.f)) return TRN_E_UNSUPPORTED;
    const int64_t D = d->head_dim;
    if (d->q_stride_s < D || d->k_stride_s < D) return TRN_E_STRIDE;
    if (need_v && (d->v_stride_s < D || d->o_stride_s < D)) return TRN_E_STRIDE;
    const int64_t st[] = {d->q_stride_b, d->q_stride_h, d->q_stride_s, d->k_stride_b, d->k_stride_h, d->k_stride_s};
    for (int64_t x : st) if (x < 0 || !pitch16(x, 2)) return TRN_E_ALIGN;
    if (need_v) {
        const int64_t sv[] = {d->v_stride_b, d->v_stride_h, d->v_stride_s, d->o_stride_b, d->o_stride_h, d->o_stride_s};
        for (int64_t x : sv) if (x < 0 || !pitch16(x, 2)) return TRN_E_ALIGN;
    }
    return TRN_OK;
}

}  // namespace trn

namespace trn {
// Workgroup shape of the forward kernel with score perturbation (us; W = workgroups of 128 queries).
//  Narrow  the general case: two workgroups of four waves per CU.
//  Split   eight waves on 128 queries halve the longest walk of a causal triangle that fills the chip once at most, for a
//          merge of 2 - 3 us.  Narrow / split: 32 heads of 128: 600 keys 22.7 / 22.3, 1250 43.0 / 39.8, 1501 (fp16) 46.4 /
//          41.9, 1600 61.6 / 58.9, 1800 (fp16) 60.6 / 58.4; 8 heads 2489 64.8 / 57.0, 4000 (fp16) 96 / 82; 2 x 8 heads, 1500
//          42.1 / 37.1; 16 heads of 64: 1100 (fp16) 26.8 / 22.4, 2500 (fp16) 55.5 / 43.1, 4034 (fp16) 115 / 90; 32 heads of
//          64, 1100 29.9 / 27.9, 2000 76 / 72.  Not where many heads bring many short walks, which even out by themselves:
//          40 heads of 128, 1200 keys (W = 400) 45.0 / 47.6, 64 heads, 700 (384) 26.6 / 33.7, 32 heads, 2048 (512) 109 / 125;
//          71 heads of 64: 400 (284) 14.7 / 17.9, 700 (426) 21.6 / 26.6.  (A query tile may then hold queries that see no
//          key of the second group's first tile only if it begins inside one: hence as many queries as keys.)
//  Wide    256 queries per K/V stage.  Unmasked, from one workgroup per CU.  Causal, where workgroups differ in length:
//          with head_dim 128 from 384 workgroups of at least six tiles per head; fewer waste too much of the last one, and
//          head_dim 64 prefers the finer grid throughout.  Narrow / wide: 32 heads of 128: 4096 keys 257 / 244, 4096 (fp16)
//          231 / 217, 3500 (fp16) 182 / 165, 3107 188 / 175, 3072 149 / 153, 2 x 1706 124 / 114, but 2560 (320) 107 / 117;
//          6 x 8 heads, 2048 122 / 131; 71 heads of 64, 2048 151 / 158.
static NoiseShape noise_shape(const trn_attn_desc* d) {
    const int64_t bh = (int64_t)d->batch * d->n_q_heads, n128 = ((int64_t)d->seq_q + 127) / 128, W = n128 * bh;
    const int64_t n256 = ((int64_t)d->seq_q + 255) / 256;
    if (d->causal && d->seq_q == d->seq_kv) {
        const bool split = d->head_dim == 128 ? (W <= 256 ? n128 >= 5 : bh <= 32 && n128 >= 9 && W < 512) : n128 >= 9 && W <= 512;
        if (split) return NoiseShape::Split;
    }
    const bool wide = d->causal ? d->head_dim == 128 && n256 >= 6 && n256 * bh >= 384 : n256 * bh >= 256;
    return wide ? NoiseShape::Wide : NoiseShape::Narrow;
}

// The non-temporal hint for the noise: its lines then don't push K, V and Q out of the L2s, and the last-level cache (256 MB)
// is not filled with what it cannot keep until the statistics read it again.  For that the rows have to lie on whole lines
// (elsewhere a line belongs to two row pieces and would be fetched twice) and the visible noise must be more than that cache
// holds for the second pass.  us, forward + statistics, without / with: 32 heads of 128: 4096 keys 253 + 215 / 244 + 190, 2560
// 114 + 102 / 107 + 94, 1792 (206 MB) 73 + 43 / 63 + 45; 71 heads of 64, 1536 83 + 73 / 77 + 70; but 1024 keys (67 MB) 35 + 21
// / 36 + 25, and rows off the lines: 3107 keys 175 + 149 / 219 + 160.
bool noise_streams(const trn_attn_desc* d, const void* noise, bool n16) {
    if (!noise || n16 || (reinterpret_cast<uintptr_t>(noise) & 127u)) return false;
    if ((d->noise_stride_s & 31) || (d->noise_stride_h & 31) || (d->noise_stride_b & 31)) return false;
    const int64_t per_head = d->causal ? (int64_t)d->seq_q * (2 * (int64_t)d->seq_kv - d->seq_q) * 2 : (int64_t)d->seq_q * d->seq_kv * 4;
    return (int64_t)d->batch * d->n_q_heads * per_head >= (int64_t)192 << 20;
}
}  // namespace trn

extern "C" int64_t trn_attn_workspace_bytes(const trn_attn_desc* d) {
    using namespace trn;
    if (!d || validate_attn(d, true) != TRN_OK) return 0;
    return attn_decode_workspace_bytes(d->batch, d->n_q_heads, d->seq_q, d->seq_kv, d->head_dim);
}

extern "C" int64_t trn_attn_chunk_workspace_bytes(const trn_attn_desc* d) {
    using namespace trn;
    if (!d || validate_attn(d, true) != TRN_OK) return 0;
    if (d->seq_q <= 32) return attn_few_query_workspace_bytes(d->batch, d->n_q_heads, d->n_kv_heads, d->seq_q, d->seq_kv, d->head_dim);
    return attn_share_workspace_bytes(d->batch, d->n_q_heads, d->seq_q, d->seq_kv, d->head_dim);
}

extern "C" const char* trn_attn_fwd_kernel_name(const trn_attn_desc* d, int32_t with_noise) {
    using namespace trn;
    if (!d || validate_attn(d, true) != TRN_OK) return "";
    const bool d128 = d->head_dim == 128;
    if (attn_decode_suits(d->batch, d->n_q_heads, d->seq_q, d->seq_kv, d->head_dim, d->causal != 0, with_noise != 0))
        return attn_decode_kernel_name(d->batch, d->n_q_heads, d->seq_q, d->seq_kv, d->head_dim, with_noise != 0);
    if (!with_noise) return attn_fwd16_kernel_name(d->head_dim, attn_fwd16_shape(d->batch, d->n_q_heads, d->seq_q, d->seq_kv, d->head_dim, d->causal != 0));
    trn_attn_desc n = *d;
    if (!n.noise_stride_s && !n.noise_stride_h && !n.noise_stride_b) {       // (no noise described: a contiguous one)
        n.noise_stride_s = n.seq_kv; n.noise_stride_h = n.seq_q * n.noise_stride_s; n.noise_stride_b = n.n_q_heads * n.noise_stride_h;
    }
    const bool stream = noise_streams(&n, reinterpret_cast<const void*>((uintptr_t)(with_noise == 2 ? 16 : 128)), false);
    const NoiseShape shape = noise_shape(d);
    if (shape == NoiseShape::Split) {
        if (d128) return stream ? "trn::attn_fwd_split_kernel<128, false, true>" : "trn::attn_fwd_split_kernel<128, false, false>";
        return stream ? "trn::attn_fwd_split_kernel<64, false, true>" : "trn::attn_fwd_split_kernel<64, false, false>";
    }
    const bool wide = shape == NoiseShape::Wide, usual = stream == (d128 && wide);
    if (d128) return wide ? (usual ? "trn::attn_fwd_kernel<128, 8, true>" : "trn::attn_fwd_kernel<128, 8, false>")
                          : (usual ? "trn::attn_fwd_kernel<128, 4, true>" : "trn::attn_fwd_kernel<128, 4, false>");
    return wide ? (usual ? "trn::attn_fwd_kernel<64, 8, true>" : "trn::attn_fwd_kernel<64, 8, false>")
                : (usual ? "trn::attn_fwd_kernel<64, 4, true>" : "trn::attn_fwd_kernel<64, 4, false>");
}

extern "C" int trn_attn_fwd_f16(const trn_attn_desc* d, const void* q, const void* k, const void* v, void* o,
                                float* lse, const void* gamma_q, const float* noise, float* lse_pert,
                                void* stream) {
    return trn_attn_fwd_ws_f16(d, q, k, v, o, lse, gamma_q, noise, lse_pert, nullptr, 0, stream);
}

extern "C" int trn_attn_fwd_ws_f16(const trn_attn_desc* d, const void* q, const void* k, const void* v, void* o,
                                   float* lse, const void* gamma_q, const float* noise, float* lse_pert,
                                   void* workspace, int64_t workspace_bytes, void* stream) {
    return trn::attn_forward(d, q, k, v, o, lse, gamma_q, noise, lse_pert, workspace, workspace_bytes, nullptr, nullptr, stream);
}

extern "C" int trn_attn_colstats_f16(const trn_attn_desc* d, const void* q, const void* k, const float* lse,
                                     const float* noise, float* out_sum, float* out_sumsq, void* stream);

extern "C" int trn_attn_fwd_probs_f16(const trn_attn_desc* d, const void* q, const void* k, const void* v, void* o,
                                      float* lse, const float* noise, float* lse_pert,
                                      float* out_probs, float* out_sum, void* stream) {
    using namespace trn;
    if (!d || !out_probs) return TRN_E_NULL;
    if (d->seq_q > 32) return TRN_E_UNSUPPORTED;     // the un-reduced matrix is a decode-shape output
    if (d->q_norm) return TRN_E_UNSUPPORTED;
    return attn_forward(d, q, k, v, o, lse, nullptr, noise, lse_pert, nullptr, 0, out_sum, nullptr, stream, out_probs);
}

extern "C" int trn_attn_fwd_stats_f16(const trn_attn_desc* d, const void* q, const void* k, const void* v, void* o,
                                      float* lse, const void* gamma_q, const float* noise, float* lse_pert,
                                      float* out_sum, float* out_sumsq, void* stream) {
    using namespace trn;
    if (!d) return TRN_E_NULL;
    if (!out_sum && !out_sumsq) return TRN_E_NULL;
    if (d->q_norm) return TRN_E_UNSUPPORTED;     // the statistics pass takes the queries as given
    // a handful of queries per head: the statistics are a second sweep inside the same kernel
    if (d->seq_q <= 32) return attn_forward(d, q, k, v, o, lse, gamma_q, noise, lse_pert, nullptr, 0, out_sum, out_sumsq, stream);
    // otherwise two launches; the second needs the first one's row normalisers
    float* rows = noise ? lse_pert : lse;
    if (!rows) return TRN_E_NULL;
    const int st = attn_forward(d, q, k, v, o, lse, gamma_q, noise, lse_pert, nullptr, 0, nullptr, nullptr, stream);
    if (st != TRN_OK) return st;
    return trn_attn_colstats_f16(d, q, k, rows, noise, out_sum, out_sumsq, stream);
}

// (attention_with_stats and its C entry split where heads x head_dim is at most 2048, from 8 keys per unit of it and 4096 on;
// the key scores of the modules where their own rule says so)
extern "C" int64_t trn_attn_stats_workspace_bytes(const trn_attn_desc* d) {
    const int64_t need = trn_attn_workspace_bytes(d);
    if (need == 0) return 0;
    const int64_t per_key = (int64_t)d->batch * d->n_q_heads * d->head_dim;
    return per_key <= 2048 && d->seq_kv >= (8 * per_key > 4096 ? 8 * per_key : 4096) ? need : 0;
}

extern "C" int64_t trn_attn_key_scores_workspace_bytes(const trn_attn_desc* d, int32_t with_noise) {
    using namespace trn;
    if (!d || validate_attn(d, true) != TRN_OK) return 0;
    // a chunk of more than 32 queries without noise: its forward shares out the keys as it does without the statistics
    if (d->seq_q > 32 && with_noise) return noise_strips_workspace_bytes(d, with_noise);
    if (d->seq_q > 32) return attn_share_workspace_bytes(d->batch, d->n_q_heads, d->seq_q, d->seq_kv, d->head_dim);
    return attn_decode_stats_workspace_bytes(d->batch, d->n_q_heads, d->seq_q, d->seq_kv, d->head_dim, with_noise != 0);
}

extern "C" int trn_attn_fwd_stats_ws_f16(const trn_attn_desc* d, const void* q, const void* k, const void* v, void* o,
                                         float* lse, const void* gamma_q, const float* noise, float* lse_pert,
                                         float* out_sum, float* out_sumsq, void* workspace, int64_t workspace_bytes,
                                         void* stream) {
    using namespace trn;
    if (!d) return TRN_E_NULL;
    if (!out_sum && !out_sumsq) return TRN_E_NULL;
    if (d->q_norm) return TRN_E_UNSUPPORTED;
    if (workspace && ((reinterpret_cast<uintptr_t>(workspace) & 255u) != 0 || workspace_bytes < 0)) return TRN_E_ALIGN;
    // Few queries on a long cache: the keys are split over workgroups (which needs the workspace), and a second launch merges
    // them and sums up the statistics -- in calls that ask for the row normalisers.  Everything else runs as
    // trn_attn_fwd_stats_f16.
    const int64_t need = trn_attn_stats_workspace_bytes(d);
    float* rows = noise ? lse_pert : lse;
    if (workspace && need > 0 && workspace_bytes >= need && rows)
        return attn_forward(d, q, k, v, o, lse, gamma_q, noise, lse_pert, workspace, workspace_bytes, out_sum, out_sumsq, stream);
    return trn_attn_fwd_stats_f16(d, q, k, v, o, lse, gamma_q, noise, lse_pert, out_sum, out_sumsq, stream);
}

extern "C" int trn_attn_fwd_stats_half_f16(const trn_attn_desc* d, const void* q, const void* k, const void* v, void* o,
                                           float* lse, const void* gamma_q, const void* noise, float* lse_pert,
                                           void* out_sum, void* out_sumsq, void* stream) {
    using namespace trn;
    if (!d) return TRN_E_NULL;
    if (!out_sum && !out_sumsq) return TRN_E_NULL;
    if (d->q_norm || d->seq_q > 32) return TRN_E_UNSUPPORTED;
    if (noise && ((reinterpret_cast<uintptr_t>(noise) & 7u) || (d->noise_stride_s & 3) || (d->noise_stride_h & 3) || (d->noise_stride_b & 3)))
        return TRN_E_ALIGN;
    return attn_forward(d, q, k, v, o, lse, gamma_q, static_cast<const float*>(noise), lse_pert, nullptr, 0,
                        static_cast<float*>(out_sum), static_cast<float*>(out_sumsq), stream, nullptr, true, true);
}

extern "C" int trn_attn_key_scores_f16(const trn_attn_desc* d, const void* q, const void* k, const void* v, void* o,
                                       const void* noise, int32_t noise_half, float* rows, void* out1, void* out2,
                                       int32_t out_half, int32_t mean_std, void* workspace, int64_t workspace_bytes,
                                       void* stream) {
    using namespace trn;
    if (!d || !rows || (!out1 && !out2) || (mean_std && !(out1 && out2))) return TRN_E_NULL;
    if (d->q_norm || (mean_std && noise)) return TRN_E_UNSUPPORTED;
    const float* n = static_cast<const float*>(noise);
    float *lse = noise ? nullptr : rows, *lse_pert = noise ? rows : nullptr, *s1 = static_cast<float*>(out1), *s2 = static_cast<float*>(out2);
    const bool n16 = noise && noise_half, s16 = out_half != 0;
    // A workspace that cannot be used is as good as none: the keys are not split then.  Misaligned ones of the size and problems
    // that trn_attn_stats_workspace_bytes() names have always been refused.
    if (workspace && ((reinterpret_cast<uintptr_t>(workspace) & 255u) || workspace_bytes < 0)) {
        const int64_t named = trn_attn_stats_workspace_bytes(d);
        if (named > 0 && workspace_bytes >= named) return TRN_E_ALIGN;
        workspace = nullptr; workspace_bytes = 0;
    }
    // a handful of queries per head: the statistics are part of the same kernel, or of the launch that merges the key shares
    if (d->seq_q <= 32 && !mean_std)
        return attn_forward(d, q, k, v, o, lse, nullptr, n, lse_pert, workspace, workspace_bytes, s1, s2, stream, nullptr, n16, s16, true);
    // (a problem that the second launch refuses is refused before the first has written anything)
    int st = attn_colstats_check(d, q, k, rows, n, s1, s2, n16, true);
    if (st != TRN_OK) return st;
    if (attn_short_suits(d->seq_q, d->seq_kv))
        return attn_forward(d, q, k, v, o, lse, nullptr, n, lse_pert, nullptr, 0, s1, s2, stream, nullptr, n16, s16, true, false, nullptr, 0.f, mean_std != 0);
    // The scores of a prompt in one pass over the noise, and its attention, which needs none, on the kernels without it (the queries
    // as given, as the forward with noise takes them)
    const int64_t parts = n && s1 && !s2 && noise_strip_slots(d, n16) > 0 ? noise_strips_workspace_bytes(d, n16 ? 2 : 3) : -1;
    if (parts == 0 || (parts > 0 && workspace && workspace_bytes >= parts)) {
        // (in this order, so that the attention takes the sums of a head's workgroups along, 3 us as a launch of their own; what the attention refuses is
        // refused before anything is written)
        if (st = attn_forward(d, q, k, v, o, nullptr, nullptr, nullptr, nullptr, nullptr, 0, nullptr, nullptr, nullptr, nullptr, false, false, false, false,
                              nullptr, 0.f, false, true, nullptr, true); st != TRN_OK) return st;
        SlotSums sums;
        if (launch_noise_strips(d, q, k, noise, n16, rows, out1, s16, workspace, sums, (hipStream_t)stream) != hipSuccess) return TRN_E_LAUNCH;
        return attn_forward(d, q, k, v, o, nullptr, nullptr, nullptr, nullptr, nullptr, 0, nullptr, nullptr, stream, nullptr, false, false, false, false,
                            nullptr, 0.f, false, true, &sums);
    }
    // mean and deviation of a handful of queries: by the launch that merges the key shares; elsewhere the workspace stays
    // out of it (the plain attention would split the keys by counters in it that have to be zero)
    if (d->seq_q <= 32) {
        if (workspace && attn_decode_stat_shares(d->batch, d->n_q_heads, d->n_kv_heads, d->seq_q, d->seq_kv, d->head_dim, false, workspace_bytes) > 0)
            return attn_forward(d, q, k, v, o, lse, nullptr, n, lse_pert, workspace, workspace_bytes, s1, s2, stream, nullptr, n16, s16, true, false, nullptr, 0.f, true);
        workspace = nullptr; workspace_bytes = 0;
    }
    st = attn_forward(d, q, k, v, o, lse, nullptr, n, lse_pert, workspace, workspace_bytes, nullptr, nullptr, stream, nullptr, n16, false, true);
    if (st != TRN_OK) return st;
    return attn_colstats(d, q, k, rows, n, s1, s2, mean_std ? 1 : 0, stream, n16, s16, true);
}

// Whether the attention launch takes the norm of the keys along (it needs no workspace then).
static bool norms_keys(const trn_attn_desc* d) {
    return trn::attn_decode_norms_keys(d->batch, d->n_q_heads, d->seq_q, d->seq_kv, d->head_dim);
}

extern "C" int64_t trn_attn_qknorm_workspace_bytes(const trn_attn_desc* d) {
    using namespace trn;
    if (!d || validate_attn(d, true) != TRN_OK || norms_keys(d)) return 0;
    return (int64_t)d->batch * d->n_kv_heads * d->seq_kv * d->head_dim * 2;
}

extern "C" int trn_attn_qknorm_f16(const trn_attn_desc* d, const void* q, const void* k, const void* v, void* o,
                                   const void* gamma_q, const void* gamma_k, float k_eps, void* k_norm, void* stream) {
    using namespace trn;
    if (!d || !k) return TRN_E_NULL;
    const int st = validate_attn(d, true);
    if (st != TRN_OK) return st;
    if (!aligned16(k) || (gamma_k && !aligned16(gamma_k))) return TRN_E_ALIGN;
    if (norms_keys(d))
        return attn_forward(d, q, k, v, o, nullptr, gamma_q, nullptr, nullptr, nullptr, 0, nullptr, nullptr, stream, nullptr,
                            false, false, false, true, gamma_k, k_eps);
    if (!k_norm) return TRN_E_NULL;
    // (the stride from one head's keys to the next, batch by batch; a single head has none of its own)
    const int64_t head = d->n_kv_heads == 1 ? d->k_stride_b : d->k_stride_h;
    if (d->batch > 1 && d->k_stride_b != d->n_kv_heads * head) return TRN_E_STRIDE;
    const int64_t rows = d->seq_kv, D = d->head_dim;
    if (const int e = trn_rmsnorm_f16(k, gamma_k, k_norm, (int64_t)d->batch * d->n_kv_heads, rows, D, head, d->k_stride_s,
                                      rows * D, D, 0, k_eps, stream); e != TRN_OK) return e;
    trn_attn_desc n = *d;
    n.k_stride_b = d->n_kv_heads * rows * D; n.k_stride_h = rows * D; n.k_stride_s = D;
    return attn_forward(&n, q, k_norm, v, o, nullptr, gamma_q, nullptr, nullptr, nullptr, 0, nullptr, nullptr, stream);
}

int trn::attn_forward(const trn_attn_desc* d, const void* q, const void* k, const void* v, void* o, float* lse,
                             const void* gamma_q, const float* noise, float* lse_pert, void* workspace,
                             int64_t workspace_bytes, float* col_sum, float* col_sumsq, void* stream, float* probs,
                             bool n16, bool s16, bool any_pitch, bool k_norm, const void* gamma_k, float k_eps, bool mean_std, bool given_q,
                             const SlotSums* sums, bool check_only) {
    if (workspace && ((reinterpret_cast<uintptr_t>(workspace) & 255u) != 0 || workspace_bytes < 0)) return TRN_E_ALIGN;
    if (!d || !q || !k || !v || !o) return TRN_E_NULL;
    if (noise && !lse_pert) return TRN_E_NULL;
    int st = validate_attn(d, true);
    if (st != TRN_OK) return st;
    if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(o) || (gamma_q && !aligned16(gamma_q)))
        return TRN_E_ALIGN;
    if (noise) {
        if (!(d->tau > 0.f)) return TRN_E_UNSUPPORTED;
        if (d->noise_stride_s < d->seq_kv) return TRN_E_STRIDE;
        // one head's noise is addressed with 32-bit byte offsets
        if ((int64_t)d->seq_q * d->noise_stride_s * 4 + 1024 > 0x7fffffffLL) return TRN_E_UNSUPPORTED;
        if (n16 || any_pitch) {   // fp16: whole dwords around the rows are fetched and shifted; fp32: 16-byte loads on any dword
            if (reinterpret_cast<uintptr_t>(noise) & (n16 ? 1u : 3u)) return TRN_E_ALIGN;
        } else if (!aligned16(noise) || !pitch16(d->noise_stride_s, 4) || !pitch16(d->noise_stride_h, 4) ||
                   !pitch16(d->noise_stride_b, 4))
            return TRN_E_ALIGN;
    }
    AttnArgs a;
    a.q = (const half_t*)q; a.k = (const half_t*)k; a.v = (const half_t*)v; a.o = (half_t*)o;
    a.lse = lse; a.gamma_q = (const half_t*)gamma_q; a.noise = noise; a.lse_pert = lse_pert;
    a.B = d->batch; a.Hq = d->n_q_heads; a.Hkv = d->n_kv_heads; a.Sq = d->seq_q; a.Skv = d->seq_kv;
    a.n_qtiles = 0;   // set per tile shape at launch
    a.heads = HeadMap(a.B, a.Hq, a.Hkv);
    a.qb = d->q_stride_b; a.qh = d->q_stride_h; a.qs = d->q_stride_s;
    a.kb = d->k_stride_b; a.kh = d->k_stride_h; a.ks = d->k_stride_s;
    a.vb = d->v_stride_b; a.vh = d->v_stride_h; a.vs = d->v_stride_s;
    a.ob = d->o_stride_b; a.oh = d->o_stride_h; a.os = d->o_stride_s;
    a.nb = d->noise_stride_b; a.nh = d->noise_stride_h; a.ns = d->noise_stride_s;
    a.c1 = d->scale * kLog2e;
    const float tau = noise ? d->tau : 1.f;
    a.c2 = d->scale * kLog2e / tau; a.c3 = kLog2e / tau;
    a.q_eps = d->q_norm_eps; a.causal = d->causal ? 1 : 0; a.q_norm = d->q_norm ? 1 : 0;
    a.gamma_k = (const half_t*)gamma_k; a.k_eps = k_eps; a.k_norm = k_norm ? 1 : 0;
    a.n_split = 1; a.spread = 0; a.ws = nullptr; a.col_sum = col_sum; a.col_sumsq = col_sumsq; a.probs = probs; a.mean_std = mean_std ? 1 : 0; a.n16 = n16 ? 1 : 0; a.s16 = s16 ? 1 : 0;
    a.o_nt = outputs_stream((int64_t)d->batch * d->n_q_heads * d->seq_q, d->head_dim) ? 1 : 0;
    // K/V tiles are fetched with 32-bit buffer offsets relative to the (batch, head) base
    // (with room for the blocks the pipelines request past the end, which must stay representable to read as zeros)
    if (((int64_t)d->seq_kv + 2048) * d->k_stride_s * 2 > 0x7fffffffLL || ((int64_t)d->seq_kv + 2048) * d->v_stride_s * 2 > 0x7fffffffLL)
        return TRN_E_UNSUPPORTED;
    if (check_only) return TRN_OK;
    hipStream_t s = (hipStream_t)stream;
    hipError_t e;
    if ((col_sum || col_sumsq) && d->seq_q > 32) {
        // (what that kernel does not do: the callers see to it)
        if (!attn_short_suits(d->seq_q, d->seq_kv) || d->q_norm || k_norm || probs) return TRN_E_UNSUPPORTED;
        return launch_attn_short(a, d->head_dim, s) == hipSuccess ? TRN_OK : TRN_E_LAUNCH;
    }
    // a chunk of queries on a long cache, with the workspace for it: the keys shared out over workgroups
    if (workspace && !noise && !col_sum && !col_sumsq && !probs) {
        const int64_t need = attn_share_workspace_bytes(d->batch, d->n_q_heads, d->seq_q, d->seq_kv, d->head_dim);
        if (need > 0 && workspace_bytes >= need) {
            a.ws = static_cast<float*>(workspace);
            return launch_attn_shares(a, d->head_dim, s) == hipSuccess ? TRN_OK : TRN_E_LAUNCH;
        }
    }
    // few queries per head (decode), or few query tiles in all: one workgroup per head and 32 queries, its waves split the keys
    if (attn_decode_suits(d->batch, d->n_q_heads, d->seq_q, d->seq_kv, d->head_dim, d->causal && !(sums && sums->n_slots > 0), noise != nullptr)) {
        if (sums && sums->n_slots > 0 && launch_add_slots(*sums, s) != hipSuccess) return TRN_E_LAUNCH;
        return launch_attn_decode(a, d->head_dim, workspace, workspace_bytes, s) == hipSuccess ? TRN_OK : TRN_E_LAUNCH;
    }
    if (sums) a.sums = *sums; else a.sums.n_slots = 0;
    // Without score perturbation: the 16x16x32 kernel, in the workgroup shape its launcher's rule picks.
    if (!noise)
        return launch_attn_fwd16(a, d->head_dim, attn_fwd16_shape(d->batch, d->n_q_heads, d->seq_q, d->seq_kv, d->head_dim, d->causal != 0), given_q, s) == hipSuccess ? TRN_OK : TRN_E_LAUNCH;
    // With it: the shape of noise_shape().
    const NoiseShape shape = noise_shape(d);
    const bool stream_noise = noise_streams(d, noise, n16);
    e = d->head_dim == 128 ? launch_fwd<128>(a, shape, stream_noise, s) : launch_fwd<64>(a, shape, stream_noise, s);
    return e == hipSuccess ? TRN_OK : TRN_E_LAUNCH;
}
