// Flash attention forward for gfx950 on the 16x16x32 MFMA: O = softmax(scale * Q K^T [+causal]) V, GQA/MQA,
// head_dim 64/128, no score perturbation (that variant stays on the 32x32x16 kernel in attn_fwd.hip).
//
// Why a second kernel for the same arithmetic: at these shapes the chip is power-limited, and per flop the
// 16x16x32 instruction reads and writes half as many accumulator registers as the 32x32x16 one (a 16x16 fp32 block
// per 16 K flop against a 32x32 block per 32 K flop).  Issued back to back on random operands it sustains about
// 17 % more flops at the board's power limit; whatever part of that survives the softmax work is free.
//
// Formulation (transposed, as in attn_fwd.hip).  A wave owns 32 queries as two blocks of 16 (qb); lane l = 16 g + n
// holds queries 16 qb + n.  Per 32-key block, split in two halves of 16 keys (kb):
//     S^T(kb, qb)[key][query] = K[16 kb + key][:] . Q[16 qb + query][:]   A = K rows from LDS (one 16-byte read:
//                               row n, contraction columns 32 ks + 8 g ..+7), B = Q^T in registers
//   the lane receives keys 16 kb + 4 g + 0..3 of its two queries: 8 keys per query, the other 24 sit in the
//   lanes n + 16, n + 32, n + 48.  The running max is kept equal in the four lanes of a query, and whether it must
//   rise is decided from the lane's own 8 keys (any lane of the wave over the threshold raises it for all), so the
//   common path has no cross-lane traffic at all.  Row sums come from the matrix pipe (an all-ones A operand).
//     O^T(db, qb)[d][query] += V^T[16 db + d][slot] * P^T[slot][query]   one MFMA per 32-key block (K = 32)
//   contraction slot 8 g + j of a lane is key 4 g + j (j < 4) or 16 + 4 g + (j - 4): exactly the keys whose
//   scores the lane holds, so P goes from the S^T accumulators to the B operand without leaving the lane, and the
//   A operand takes its two transposing reads from rows 4 g .. and 16 + 4 g .. of the V stage.
// The exponent comes out of the matrix pipe ready-made: Q is multiplied by scale * log2(e) once in the prologue, and
// every score chain starts from the accumulator {-m} instead of zero, so S^T arrives as s - m and the softmax costs
// one v_exp_f32 per score and nothing else (the multiply-subtract it replaces was a quarter of the loop's vector
// instructions).  When the lazy maximum rises, the scores already in flight are shifted along with it.
// Staging (global -> LDS loads, XOR swizzle, two stages each for K and V, one barrier per 64-key tile), the grid
// and the lazy running maximum are those of attn_fwd.hip.
#include "attn.h"
#include <type_traits>

namespace trn {

// What the two groups of four waves of an eight-wave workgroup do: kPlain, the same tile of 256 queries; kPaired, two
// tiles of 128 queries from the two ends of a causal problem; kSplit, the same 128 queries, each group every other
// 64-key tile -- of 128 consecutive queries or, under a causal mask, of two tiles of 64 from the two ends (a.even) --; kShare, as kSplit on one of a.n_split shares of the keys, whose partial results a second launch merges.
enum { kPlain, kPaired, kSplit, kShare };

__device__ __forceinline__ float4_t mfma16(half8_t a, half8_t b, float4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}
// v_permlane16_swap exchanges the odd 16-lane rows of one register with the even rows of another: from two
// copies of x it leaves the values of rows {0, 0, 2, 2} and {1, 1, 3, 3}.  Followed by the 32-lane exchange this
// combines the four lanes n, n + 16, n + 32, n + 48.
__device__ __forceinline__ void swap_rows16(float& a, float& b) {
    asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
}
__device__ __forceinline__ int imax3(int a, int b, int c) { return max(max(a, b), c); }
__device__ __forceinline__ float quad_max(float x) { float a = x, b = x; swap_rows16(a, b); return half_max(fmaxf(a, b)); }
__device__ __forceinline__ float quad_sum(float x) { float a = x, b = x; swap_rows16(a, b); return half_sum(a + b); }

// XOR swizzle of the 16-byte chunk index within a stage row for this kernel's access patterns.  The LDS has 64
// banks (256 bytes per clock).  A 16-byte read is served 16 lanes at a time, and the lanes served together are
// {0-3, 12-15, 20-27}, {4-11, 16-19, 28-31} and the same plus 32 (measured: two lanes that read different addresses
// in the same bank cost a cycle exactly when both are in one of these sets); the transposing 8-byte read is served
// in halves of the wave.  (a) A K operand read has lane 16 g + n on row n at logical chunk 4 ks + g, so a set holds
// the rows {0-3, 12-15} at one chunk and the rows {4-11} at its neighbour: no two rows, one from each, may have
// swizzles that differ in bit 0 only.  (b) A transposing V read has each half of the wave on 8 consecutive rows x 2
// adjacent chunks: the swizzle without bit 0 must be distinct over those rows.  (Rows of 128 bytes: two share a
// 256-byte line, and the conditions hold per row parity.)
template <int D> __device__ __forceinline__ int swz16(int r) {
    if constexpr (D == 128) return ((r & 7) << 1) ^ ((r & 8) ? 9 : 0);       // rows 12 apart differ in bit 0 only
    else return r & 6;
}

struct Scores16 { float4_t s[2][2]; };      // [key half][query block]

#if defined(__HIP_DEVICE_COMPILE__)
// GIVEN: the queries enter the products as they are given, and the fp32 scores are multiplied by scale * log2(e) -- one FMA a score,
// behind the MFMAs of phase B, which also subtracts m (the chains start from zero then).  Q times scale * log2(e) rounded to fp16
// is another rounding of the queries: O against float64, 1024 tokens, 32 heads of 128: 3.1e-4 for N(0,1), 4.0e-4 and 6.1e-4 for queries
// twice and eight times as large, where the queries as given leave 2.5e-4, 2.5e-4 and 2.1e-4.  For KeyFormer's prompts whose noise has a
// pass of its own, as the kernel that takes the noise along does.  Whole calls, us, Q rounded / as given: 32 heads of 128, 2048 keys, fp32
// noise 127 / 129, 777 40.3 / 41.0, 1000 fp16 43.6 / 44.7; 71 of 64, 1536 fp32 114.7 / 117.3, 1100 fp16 67.6 / 68.9.
template <int D, int NW, int MODE, bool GIVEN = false>
__device__ __forceinline__ void attn_fwd16_body(const AttnArgs& a) {
    constexpr bool PAIRED = MODE == kPaired, SHARE = MODE == kShare, SPLIT = MODE == kSplit || SHARE;
    static_assert(MODE == kPlain || NW == 8, "paired query tiles and split keys are two groups of four waves");
    constexpr int GW = SPLIT ? 4 : NW;       // waves that share the K / V stages
    constexpr int KSTEP = SPLIT ? 128 : 64;  // keys from one tile of a wave to its next
    constexpr int BN = 64;       // keys per LDS stage (two 32-key blocks)
    constexpr int NS = D / 8;    // MFMA slots per phase: 2 key halves x 2 query blocks x D/32 steps of S^T; D/16 x 2 of P V
    constexpr int NKS = D / 32;  // contraction steps of S^T
    constexpr int NOP = D / 16;  // LDS operands per phase (each feeds the MFMAs of both query blocks)
    constexpr int CPR = D / 8;   // 16-byte chunks per row
    constexpr int RPI = 64 / CPR;            // stage rows covered by one wave-wide 1 KB load
    constexpr int NI = BN / (RPI * GW);      // such loads per wave per stage (K and V each)
    constexpr int NG = SPLIT ? 2 : 1;        // groups with stages of their own
    constexpr int SR = SHARE ? 32 : BN;      // keys per stage of the ring: two stages of a tile, or four of a block (see share_tile)
    __shared__ __attribute__((aligned(1024))) half_t Ks0_[NG * SR * D];
    __shared__ __attribute__((aligned(1024))) half_t Ks1_[NG * SR * D];
    __shared__ __attribute__((aligned(1024))) half_t Vs0_[NG * SR * D];
    __shared__ __attribute__((aligned(1024))) half_t Vs1_[NG * SR * D];
    __shared__ __attribute__((aligned(1024))) half_t Ks2_[SHARE ? NG * SR * D : 1];
    __shared__ __attribute__((aligned(1024))) half_t Ks3_[SHARE ? NG * SR * D : 1];
    __shared__ __attribute__((aligned(1024))) half_t Vs2_[SHARE ? NG * SR * D : 1];
    __shared__ __attribute__((aligned(1024))) half_t Vs3_[SHARE ? NG * SR * D : 1];

    const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, g4 = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int grp = SPLIT ? wave >> 2 : 0, gw = SPLIT ? wave & 3 : wave;
    half_t* const Ks0 = Ks0_ + grp * SR * D;
    half_t* const Ks1 = Ks1_ + grp * SR * D;
    half_t* const Vs0 = Vs0_ + grp * SR * D;
    half_t* const Vs1 = Vs1_ + grp * SR * D;
    // Query heads of one KV head: a group of waves is 2^pack of them times as many blocks of 32 queries (see packed_heads).
    const int pack = MODE == kPlain ? a.pack : 0, lead = gw >> pack, QW = GW >> pack;
    const int units = a.heads.all.of(blockIdx.x);
    // The shares of a query tile are consecutive; a share is a whole number of tiles, which the groups take in turns (not of pairs of
    // tiles: 4100 keys in eight shares would be seven of 640, and are eight of at most 576).
    const int share = SHARE ? units % a.n_split : 0, tile_no = SHARE ? units / a.n_split : units;
    const int share_tiles = SHARE ? ((a.Skv + BN - 1) / BN + a.n_split - 1) / a.n_split : 0;
    const int kfirst = grp * BN + share * share_tiles * BN;      // first key of this wave's first tile

    int b, kvh, g;
    a.heads.find(blockIdx.x - units * a.heads.all.d, b, kvh, g);
    if constexpr (MODE == kPlain) g = (g << pack) + (gw & ((1 << pack) - 1));
    const int head = kvh * a.heads.G + (MODE == kPlain ? min(g, a.heads.G - 1) : g);

    const int off = a.Skv - a.Sq;                       // causal: query i sees keys <= i + off
    // Query rows.  Plain mode: the workgroup owns BM consecutive queries, latest (heaviest under a causal mask) tiles
    // first.  Paired mode (NW = 8, causal, a grid too small for a second round to even out the tiles' lengths): waves
    // 0-3 own the 128-query tile h, waves 4-7 the tile n - 1 - h from the other end, so that every workgroup has the
    // same amount of work and each SIMD holds one long and one short wave.  K/V staging follows the later tile; the
    // early waves stop at their own last visible tile as they do in plain mode.
    // Split mode on two tiles of 64 (even): waves 0, 1, 6, 7 own the later one.
    const bool even = MODE == kSplit && a.even != 0;
    int q0, q_last, wq0;
    if constexpr (PAIRED) {
        const int lt = tile_no, ht = a.n_qtiles - 1 - lt;     // n_qtiles counts 128-query tiles here
        q0 = ht * 128; q_last = q0 + 127;
        wq0 = (wave < 4 ? ht : lt) * 128 + (wave & 3) * 32;
        if (wave >= 4 && lt == ht) wq0 = a.Sq;          // odd tile count: the middle one is alone (loads clamp, stores are predicated off)
    } else if (even) {              // (a SIMD has waves w and w + 4: one of the later tile and one of the earlier)
        const int ht = a.n_qtiles - 1 - tile_no;                             // n_qtiles counts 64-query tiles here
        const bool early = ((gw >> 1) ^ grp) != 0;
        q0 = ht * 64; q_last = q0 + 63;
        wq0 = (early ? tile_no : ht) * 64 + (gw & 1) * 32;
        if (early && tile_no == ht) wq0 = a.Sq;
    } else {
        q0 = (a.n_qtiles - 1 - tile_no) * (QW * 32); q_last = q0 + QW * 32 - 1;
        wq0 = q0 + lead * 32;                           // first query of this wave
        if (MODE == kPlain && g >= a.heads.G) wq0 = a.Sq;      // (no head for it)
    }
    int qrow[2];
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) qrow[qb] = wq0 + 16 * qb + n;
    half8_t qB[2][NKS];

    // ---- LDS read offsets (halfs).  K operand (ks, kb): row 16 kb + n of a 32-key block, logical chunk 4 ks + g4
    // (the swizzle depends on the row's low four bits only, so the second key half is a constant 16 rows further).
    int koff[NKS];
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) koff[ks] = n * D + (((4 * ks + g4) ^ swz16<D>(n)) << 3);
    // V^T operand db through the transposing read: in each 16-lane group lanes 4r..4r+3 supply stage row r; this
    // lane's piece is row 4 g4 + n/4 (second read: 16 rows further), head_dim columns 16 db + 4 (n%4) ..+3.
    int voff[NOP];
    {
        const int rl = 4 * g4 + (n >> 2), lc = (n & 3) >> 1, sub = (n & 1) * 4;
#pragma unroll
        for (int db = 0; db < NOP; ++db) voff[db] = rl * D + (((2 * db + lc) ^ swz16<D>(rl)) << 3) + sub;
    }

    const float4_t zero = {0.f, 0.f, 0.f, 0.f};
    float4_t oacc[NOP][2];                  // [16 head_dim columns][query block]
#pragma unroll
    for (int i = 0; i < NOP; ++i) oacc[i][0] = oacc[i][1] = zero;
    float m[2] = {-INFINITY, -INFINITY};    // reference max (log2 domain), equal in the four lanes of a query
    float4_t negm[2];                       // {-m} x 4: the initial accumulator of every score chain, so that the
                                            // scores arrive as s - m and the exponential needs no subtraction
    // Row sums come out of the matrix pipe as well: one more MFMA per query block whose A operand is all ones leaves
    // the sum of the block's (fp16-rounded) probabilities of each query in every row of a 16 x 16 accumulator.  Two
    // MFMAs per 32-key block instead of eight dot-product instructions, each of which costs two VALU issue slots.
    float4_t lacc[2] = {zero, zero};
    // Split keys under a causal mask: a query may see nothing in this group's first tiles.  Its reference then stays 0
    // with zero sums, and its first visible scores set it (any_fresh: some query of the wave is still in that state).
    bool fresh[2] = {false, false}, any_fresh = false;

    int ntiles = (a.Skv + BN - 1) / BN;
    if (a.causal) ntiles = min(ntiles, (min(q_last, a.Sq - 1) + off) / BN + 1);
    if constexpr (SHARE) ntiles = max(0, min(ntiles - share * share_tiles, share_tiles));      // of this share

    // ---- staging: direct global -> LDS loads; keys past the end read as zeros
    const __amdgpu_buffer_rsrc_t krs = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(a.k + b * a.kb + kvh * a.kh), 0, (int)(((int64_t)(a.Skv - 1) * a.ks + D) * 2), 0x00020000);
    const __amdgpu_buffer_rsrc_t vrs = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(a.v + b * a.vb + kvh * a.vh), 0, (int)(((int64_t)(a.Skv - 1) * a.vs + D) * 2), 0x00020000);
    const int st_row = gw * RPI + lane / CPR;
    const int st_chunk = (lane % CPR) ^ swz16<D>(st_row);
    const int kvo = (int)(st_row * a.ks * 2) + st_chunk * 16;
    const int vvo = (int)(st_row * a.vs * 2) + st_chunk * 16;
    const int krow_bytes = (int)(RPI * a.ks * 2), vrow_bytes = (int)(RPI * a.vs * 2);
    const int ktile_bytes = (int)(KSTEP * a.ks * 2), vtile_bytes = (int)(KSTEP * a.vs * 2);
    const int kgrp_bytes = (int)(kfirst * a.ks * 2), vgrp_bytes = (int)(kfirst * a.vs * 2);
#define TRN_FETCH_K(jt_, dst_) fetch_tile<NI, D, GW>(krs, &dst_[gw * RPI * D], kvo, kgrp_bytes + (jt_) * ktile_bytes, krow_bytes)
#define TRN_FETCH_V(jt_, dst_) fetch_tile<NI, D, GW>(vrs, &dst_[gw * RPI * D], vvo, vgrp_bytes + (jt_) * vtile_bytes, vrow_bytes)

    const int wb = wq0 + off;          // key index bound of this wave's first query
    auto needs_mask = [&](int key0) { return (key0 + 32 > a.Skv) || (a.causal && key0 + 31 > wb); };

    // Scores of a 32-key block starting at key0, just produced: keys past the end and, under a causal mask, keys
    // after the query become -inf.
    // (a constant against one bound per query: two vector instructions a score where the key's index, two comparisons and
    // their conjunction took five, and short walks mask every third tile: 4 x 777 tokens, 32 heads of 128, 32.7 -> 32.0 us;
    // 71 heads of 64, 547 tokens 10.4 -> 9.8)
    int last_key[2];        // the last key that the lane's queries see, less its first key within a block
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) last_key[qb] = min(a.Skv - 1, a.causal ? qrow[qb] + off : a.Skv - 1) - 4 * g4;
    auto mask_block = [&](Scores16& sx, int key0) __attribute__((always_inline)) {
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int qb = 0; qb < 2; ++qb)
#pragma unroll
                for (int i = 0; i < 4; ++i) sx.s[kb][qb][i] = 16 * kb + i <= last_key[qb] - key0 ? sx.s[kb][qb][i] : -INFINITY;
    };
    // The lane's maximum per query over its 8 keys of the block.
    auto block_max = [&](const Scores16& sx, float (&smax)[2]) __attribute__((always_inline)) {
#pragma unroll
        for (int qb = 0; qb < 2; ++qb) {
            const float4_t& u = sx.s[0][qb];
            const float4_t& w = sx.s[1][qb];
            smax[qb] = fmaxf(max3(u[0], u[1], u[2]), max3(u[3], w[0], w[1]));
            smax[qb] = max3(smax[qb], w[2], w[3]);
        }
    };
    // Is a rescale due?  The reference m is lazy (raised only when some score exceeds it by more than 2^8: see
    // attn_fwd.hip), the scores arrive relative to it, and the decision is wave-uniform, so only whether any of the
    // lane's 16 scores exceeds 8 matters.  For that the bit patterns will do: non-negative floats order as signed
    // integers and every negative float (masked scores included) lies below them.  One three-way integer maximum per
    // two scores, both queries of the lane together, no canonicalising of the operands (9 vector instructions per block
    // against 15 for two float maxima); the per-query maxima are formed on the rare path only.  In four pieces, one per
    // accumulator quad, so that they sit behind four different MFMAs.
    auto max_piece = [&](const Scores16& sx, int piece, int mx) __attribute__((always_inline)) {
        const float4_t& u = sx.s[piece >> 1][piece & 1];
        if (piece == 0) return max(imax3(__float_as_int(u[0]), __float_as_int(u[1]), __float_as_int(u[2])), __float_as_int(u[3]));
        mx = imax3(mx, __float_as_int(u[0]), __float_as_int(u[1]));
        return imax3(mx, __float_as_int(u[2]), __float_as_int(u[3]));
    };
    // the scores sx already in flight are relative to m: they move with it
    auto rescale = [&](Scores16& sx) __attribute__((always_inline)) {
        float smax[2];
        block_max(sx, smax);
#pragma unroll
        for (int qb = 0; qb < 2; ++qb) {
            float up = fmaxf(0.f, quad_max(smax[qb])), alpha = fast_exp2(-up);
            if constexpr (SPLIT) {      // a query that has seen no key yet: its first finite maximum is the reference
                const float qm = quad_max(smax[qb]);
                if (fresh[qb]) { up = qm == -INFINITY ? 0.f : qm; alpha = 1.f; }
                fresh[qb] = fresh[qb] && qm == -INFINITY;
            }
            sx.s[0][qb] = sx.s[0][qb] - up;
            sx.s[1][qb] = sx.s[1][qb] - up;
            negm[qb] = negm[qb] - up;                   // (in place, like the accumulators: a fresh vector here makes
                                                        // the path that skips the rescale copy it every block)
            lacc[qb] = lacc[qb] * alpha;
#pragma unroll
            for (int i = 0; i < NOP; ++i)
                oacc[i][qb] = oacc[i][qb] * alpha;      // (as one vector operation: written per element, the path that
                                                        // skips the rescale ends up copying every accumulator)
            m[qb] = m[qb] + up;
        }
        if constexpr (SPLIT) any_fresh = __builtin_amdgcn_ballot_w64(fresh[0] || fresh[1]) != 0;
    };

    bool more = true;       // shares: the block whose scores a step leaves is one of the wave's own (the stage of the block past its
                            // last is not its keys: scores from it must not move the reference)
    const half_t one = (half_t)1.f;
    const half8_t ones8 = {one, one, one, one, one, one, one, one};
    constexpr int NQ = 2;   // operand look-ahead, in operands (= 2 NQ MFMA slots; 4 measured no better, twice)
    static_assert(NOP % NQ == 0, "the operand window must divide the operands of a phase");
    half8_t ka[NQ];    // K operands of the next block's S^T, a rolling window ahead of use
    half8_t va[NQ];    // V^T operands of this block's P V, likewise
    auto load_k = [&](const half_t* Kb, int op, int reg) __attribute__((always_inline)) {       // op = 2 ks + kb
        ka[reg] = *reinterpret_cast<const half8_t*>(&Kb[(op & 1) * 16 * D + koff[op >> 1]]);
    };

    // One pipeline step for block B whose scores sc are complete, masked and reflected in m:
    //   phase A: MFMA: S^T of block B+1                  | VALU: P = exp2(sc*c1 - m), fp16, row sums
    //   phase B: MFMA: O^T += V^T P^T                    | VALU: mask + max of block B+1's scores
    // Every LDS operand feeds two consecutive MFMAs (the two query blocks); it is requested NQ operands before its
    // first use, into the register its predecessor has just vacated.  With SYNC (first block of a 64-key tile) the
    // tile hand-over sits right after the last request to the tile's own K stage, and the refills of the two stages that it
    // sets free go out one at a time behind the MFMAs of phase B.  A CU takes 64 bytes a clock from L2: requested all at once
    // behind the barrier, by all waves, 32 KB held up every wave's issue for some 500 of a tile's 2900 - 4300 clocks (32 heads
    // of 128: 4096 tokens 118.4 -> 117.2 us, 3600 107 -> 104.5, 777 16.8 -> 15.9; 71 of 64, 1574 31.6 -> 30.7).
    // MAYMASK = false: the caller knows that block B+1 needs no mask, and the test and its branch (which would sit in
    // the middle of phase B and split the slot sequence) are not compiled in.
    auto step = [&](bool masked_next, auto maymask_tag, auto sync_tag, Scores16& sc, Scores16& sn, const half_t* Vblk, const half_t* K1,
                    const half_t* K2, int key0_next, auto&& handover, auto&& refill) __attribute__((always_inline)) {
        constexpr bool SYNC = decltype(sync_tag)::value;
        constexpr bool MAYMASK = decltype(maymask_tag)::value;
        half8_t pB[2];
        auto load_v = [&](int db, int reg) __attribute__((always_inline)) {
            const half4_t lo = lds_read_tr16(Vblk + voff[db]);              // keys 4 g4 .. +3, dim 16 db + n
            const half4_t hi = lds_read_tr16(Vblk + 16 * D + voff[db]);     // keys 16 + 4 g4 .. +3
            va[reg] = half8_t{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        };
        auto exp_pair = [&](int p) __attribute__((always_inline)) {        // scores 2 (p%2), +1 of key half (p/2)%2, query block p/4
            const int qb = p >> 2, kb = (p >> 1) & 1, i0 = 2 * (p & 1);
            const float p0 = fast_exp2(sc.s[kb][qb][i0]);
            const float p1 = fast_exp2(sc.s[kb][qb][i0 + 1]);
            uint32_t u = pack_half2(p0, p1);
            asm volatile("" : "+v"(u));     // keeps the pair's work in this slot (it is otherwise sunk past the hand-over)
            const half2_t pp = __builtin_bit_cast(half2_t, u);
            pB[qb][4 * kb + i0] = pp[0]; pB[qb][4 * kb + i0 + 1] = pp[1];
        };
        // ---- phase A ----
#pragma unroll
        for (int i = 0; i < NS; ++i) {
            // (Gray order over the operand pair: from one MFMA to the next either the LDS operand or the query block
            // changes, never both -- 0.7 % of the kernel's time on N(0,1) data, where the time is the board's power)
            const int op = i >> 1, ks = op >> 1, kb = op & 1, qb = (i & 1) ^ (op & 1);
            if constexpr (SYNC) {
                if (i == NS - 2 * NQ) handover();
            }
            sn.s[kb][qb] = mfma16(ka[op % NQ], qB[qb][ks], ks == 0 ? (GIVEN ? zero : negm[qb]) : sn.s[kb][qb]);
            if (i & 1) {
                if (op + NQ < NOP) load_k(K1, op + NQ, op % NQ);
                else load_v(op + NQ - NOP, op % NQ);
            }
            if constexpr (NS == 16) { if ((i & 1) == 0) exp_pair(i >> 1); }
            else exp_pair(i);
            __builtin_amdgcn_sched_barrier(0);
        }
        // ---- phase B ----
        bool due = false;
        int mx = 0;
#pragma unroll
        for (int i = 0; i < NS; ++i) {
            const int db = i >> 1, qb = (i & 1) ^ (db & 1);
            oacc[db][qb] = mfma16(va[db % NQ], pB[qb], oacc[db][qb]);
            if (i & 1) {
                if (db + NQ < NOP) load_v(db + NQ, db % NQ);
                else load_k(K2, db + NQ - NOP, db % NQ);
            }
            if constexpr (SYNC) {
                constexpr int EVERY = NS / (2 * NI);
                static_assert(NS % (2 * NI) == 0, "the refills are dealt out evenly");
                if (i % EVERY == EVERY - 1) refill(i / EVERY);
            }
            constexpr int R0 = NS / 2 - (NS >= 16 ? 3 : 2);
            if constexpr (GIVEN) {      // the block's four quads of scores in the slots before R0, those of the last MFMAs last
                constexpr int PER = NS >= 16 ? 1 : 2, FIRST = R0 - 4 / PER;
                if (i >= FIRST && i < R0)
#pragma unroll
                    for (int u = PER * (i - FIRST); u < PER * (i - FIRST + 1); ++u)
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            sn.s[u >> 1][u & 1][e] = __builtin_fmaf(sn.s[u >> 1][u & 1][e], a.c1, negm[u & 1][0]);
            }
            if (i == R0) { if (MAYMASK && masked_next) mask_block(sn, key0_next); }
            if (i >= R0 && i < R0 + 4) mx = max_piece(sn, i - R0, mx);
            if (i == R0 + 3) due = __builtin_amdgcn_ballot_w64(mx > 0x41000000) != 0 || (SPLIT && any_fresh);       // 8.0f
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int qb = 0; qb < 2; ++qb) lacc[qb] = mfma16(ones8, pB[qb], lacc[qb]);
        if (SHARE ? due && more : due) rescale(sn);
    };

    // Shares: 32-key block B of this group's keys (two per tile) to its stage; past the share's last block nothing is read.
    const int n_blocks = 2 * ((ntiles - grp + 1) >> 1);
    auto request_k = [&](int blk, half_t* dst) __attribute__((always_inline)) {
        fetch_tile<(NI + 1) / 2, D, GW>(krs, dst + grp * SR * D + gw * RPI * D, blk < n_blocks ? kvo : 0x7ffffff0,
                                        kgrp_bytes + (blk >> 1) * ktile_bytes + (blk & 1) * (ktile_bytes / 4), krow_bytes);
    };
    auto request_v = [&](int blk, half_t* dst) __attribute__((always_inline)) {
        fetch_tile<(NI + 1) / 2, D, GW>(vrs, dst + grp * SR * D + gw * RPI * D, blk < n_blocks ? vvo : 0x7ffffff0,
                                        vgrp_bytes + (blk >> 1) * vtile_bytes + (blk & 1) * (vtile_bytes / 4), vrow_bytes);
    };

    // ---- prologue: K stages 0 and 1 and V stage 0; scores of block 0; first K operands of block 1 ----
    if constexpr (SHARE) {
        request_k(0, Ks0_); request_k(1, Ks1_);
        __builtin_amdgcn_sched_barrier(0);
    } else {
        TRN_FETCH_K(0, Ks0);
        // (paired tiles, whose walk is long, fare better with all of it in front and the order left to the compiler: 15 heads of 64, 3278 tokens 34.8 us so,
        // 36.2 with this order held; 11, 4598 47.2 / 48.2)
        if constexpr (PAIRED) { TRN_FETCH_V(0, Vs0); if (ntiles > 1) TRN_FETCH_K(1, Ks1); }
        else __builtin_amdgcn_sched_barrier(0);
    }

    // ---- Q^T B-operands: lane holds Q[qrow[qb]][32 ks + 8 g4 .. +7].  The loads go out behind the first K stage
    // fetch and all together, so that the workgroup's start-up pays one memory latency, not three in a row; the other two stages
    // behind them, for the first tile's hand-over.  us, in front of them / behind: 32 heads of 128, 300 tokens 9.3 / 8.95, 8 x 250 11.9 / 11.55,
    // 4 x 777 29.9 / 29.3; 71 of 64, 300 7.07 / 6.71, 4 x 200 7.83 / 7.54, 2048 46.4 / 46.2; but paired tiles, 2048 of 32 heads 37.8 / 38.3.
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) {
        const int qrow_ld = qrow[qb] < a.Sq ? qrow[qb] : a.Sq - 1;       // clamp loads; stores are predicated
        const half_t* qp = a.q + b * a.qb + head * a.qh + (int64_t)qrow_ld * a.qs + 8 * g4;
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) qB[qb][ks] = *reinterpret_cast<const half8_t*>(qp + ks * 32);
    }
    // (the norm's weights with them: behind the reduction each was a latency of its own: 71 heads of 64, 2048 tokens, both
    // launches 49.5 -> 48.8 us; 2 x 32 heads of 128, 1442 53.7 -> 50.6)
    half8_t gq[NKS];
    const bool q_norm = a.q_norm != 0, use_gq = q_norm && a.gamma_q;
    if (use_gq) {
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) gq[ks] = *reinterpret_cast<const half8_t*>(a.gamma_q + ks * 32 + 8 * g4);
    }
    if constexpr (!SHARE && !PAIRED) {
        __builtin_amdgcn_sched_barrier(0);
        TRN_FETCH_V(0, Vs0);
        TRN_FETCH_K(1, Ks1);    // (also of a single tile, whose hand-over waits for it: the compiler takes a conditional load for absent)
        __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (SHARE) {      // (the rest of the ring behind Q, whose wait would otherwise be for all of it)
        __builtin_amdgcn_sched_barrier(0);
        request_v(0, Vs0_); request_k(2, Ks2_); request_v(1, Vs1_); request_k(3, Ks3_); request_v(2, Vs2_);
        __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) {
        if (q_norm) {   // fused per-head RMSNorm of the query row (the rest of the row is in the lanes n + 16, + 32, + 48)
            float ss = 0.f;
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
                for (int e = 0; e < 8; ++e) { float f = (float)qB[qb][ks][e]; ss += f * f; }
            ss = quad_sum(ss);
            const float rstd = 1.0f / __builtin_sqrtf(ss / (float)D + a.q_eps);
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    float y = (float)qB[qb][ks][e] * rstd;
                    if (use_gq) y = (float)gq[ks][e] * y;
                    qB[qb][ks][e] = (half_t)y;
                }
            }
        }
        // the softmax scale and log2(e) go into Q once, so that the scores leave the matrix pipe ready for exp2
        if constexpr (!GIVEN)
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
            for (int e = 0; e < 8; ++e) qB[qb][ks][e] = (half_t)((float)qB[qb][ks][e] * a.c1);
    }

    if constexpr (SHARE) {
        constexpr int kBehind = 5 * NI / 2;             // K blocks 0 and 1 have landed
        __builtin_amdgcn_s_waitcnt(0x0070 | (kBehind & 15) | ((kBehind >> 4) << 14));
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
    } else {
        constexpr int kBehind = PAIRED ? 0 : 2 * NI;    // K stage 0 has landed
        __builtin_amdgcn_s_waitcnt(0x0f70 | (kBehind & 15) | ((kBehind >> 4) << 14));
        if constexpr (PAIRED) __syncthreads();
        else {
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
        }
    }

    Scores16 sA, sB;                        // scores of the current / next 32-key block (ping-pong)
    {
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
                const half8_t k0 = *reinterpret_cast<const half8_t*>(&Ks0[kb * 16 * D + koff[ks]]);
#pragma unroll
                for (int qb = 0; qb < 2; ++qb) sA.s[kb][qb] = mfma16(k0, qB[qb][ks], ks == 0 ? zero : sA.s[kb][qb]);
            }
#pragma unroll
        for (int i = 0; i < NQ; ++i) load_k(SHARE ? Ks1 : Ks0 + 32 * D, i, i);
        // block 0 sets the reference outright (every query sees key 0, so it is finite from here on)
        if constexpr (GIVEN)
#pragma unroll
            for (int i = 0; i < 4; ++i) sA.s[i >> 1][i & 1] = sA.s[i >> 1][i & 1] * a.c1;
        float smax[2];
        mask_block(sA, kfirst);
        block_max(sA, smax);
#pragma unroll
        for (int qb = 0; qb < 2; ++qb) {
            m[qb] = quad_max(smax[qb]);
            if constexpr (SPLIT) { fresh[qb] = m[qb] == -INFINITY; m[qb] = fresh[qb] ? 0.f : m[qb]; }
            negm[qb] = float4_t{-m[qb], -m[qb], -m[qb], -m[qb]};
            sA.s[0][qb] = sA.s[0][qb] - m[qb];
            sA.s[1][qb] = sA.s[1][qb] - m[qb];
        }
        if constexpr (SPLIT) any_fresh = __builtin_amdgcn_ballot_w64(fresh[0] || fresh[1]) != 0;
    }

    // One 64-key tile jt.  Kc = its own K stage (block 1 still has operands to give), Kn = the next tile's
    // K stage, Vc = its V stage, Vn = the other V stage.
    auto tile = [&](auto maymask_tag, int jt, half_t* Kc, const half_t* Kn, const half_t* Vc, half_t* Vn) __attribute__((always_inline)) {
        const int kv0 = kfirst + jt * KSTEP;
        // (unconditional: tiles past the end of the keys read as zeros into stages nobody reads, and the
        // hand-over stays free of branches)
        auto refill = [&](int i) __attribute__((always_inline)) {
            if (i < NI) fetch_piece<D, GW>(vrs, &Vn[gw * RPI * D], vvo, vgrp_bytes + (jt + 1) * vtile_bytes, vrow_bytes, i);
            else fetch_piece<D, GW>(krs, &Kc[gw * RPI * D], kvo, kgrp_bytes + (jt + 2) * ktile_bytes, krow_bytes, i - NI);
        };
        auto handover = [&]() __attribute__((always_inline)) {
            __builtin_amdgcn_s_waitcnt(0x0f70);   // this wave's share of stages Kn and Vc is in LDS
            __syncthreads();                      // ... and everyone's; Kc and Vn have had their last readers
        };
        auto none = [&]() __attribute__((always_inline)) {};
        auto none1 = [&](int) __attribute__((always_inline)) {};
        // (Past the last tile a K stage holds stale rows; scores computed from them are masked away.)
        step(needs_mask(kv0 + 32), maymask_tag, std::true_type{}, sA, sB, Vc, Kc + 32 * D, Kn, kv0 + 32, handover, refill);
        step(needs_mask(kv0 + KSTEP), maymask_tag, std::false_type{}, sB, sA, Vc + 32 * D, Kn, Kn + 32 * D, kv0 + KSTEP, none, none1);
    };
    // Tile jt of a share: K0 .. K3 and V0 .. V3 are the ring's stages from the tile's first block on.  What bounds it is how much is
    // under way from HBM: with the two stages of 64 keys above all of it had to land before the next was asked for, a tile of
    // 64 KB every 3 - 4 us.  Here block B's hand-over asks for V of block B + 3 and K of block B + 5, into the stages that block
    // B - 1 and block B + 1 have just vacated, and waits for what the one three blocks ago asked for.
    // us, two stages and shares of whole pairs of tiles / ring and shares of single tiles, without the merge: 32 heads of 128: 100
    // queries on 4.1 k keys 25.2 / 19.4, 128 on 3.2 k 22.7 / 18.3, 40 on 3.1 k 17.5 / 14.8, 128 on 8.1 k 38.5 / 33.5, 50 on 16 k
    // 52.2 / 50.4; 8 of 128: 100 on 8.1 k 16.6 / 16.4, 128 on 16 k 23.7 / 23.1; 71 of 64: 40 on 6 k 26.7 / 24.2, 64 on 6 k 27.4 / 24.7,
    // 128 on 3.1 k 20.0 / 17.0, 100 on 2.7 k 17.8 / 15.7; 16 of 64, three tiles a group at most: 60 on 4.3 k 9.8 / 9.9, 5.1 k 9.5 /
    // 10.1; 12 k 13.7 / 13.7.  With the merge, K and V out of the caches: 100 on 4.1 k 26.4 / 25.2, 128 on 8.1 k 32.0 / 32.3, 8 heads of 128, 100 on
    // 3.4 k 19.4 / 17.8, 71 of 64, 64 on 6 k 32.4 / 29.9, 100 on 2.7 k 22.1 / 21.5, 16 of 64, 100 on 4.1 k 16.3 / 15.6, 40 on 4.1 k 14.0 / 14.4.
    auto share_handover = [&](int blk, half_t* Kf, half_t* Vf) __attribute__((always_inline)) {
        constexpr int kBehind = 2 * NI;      // V of blk and K of blk + 2 have landed: behind them only two hand-overs' requests
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(0x0070 | (kBehind & 15) | ((kBehind >> 4) << 14));      // lgkmcnt(0): the vacated stages have been read
        __builtin_amdgcn_s_barrier();        // (a bare barrier: the loads in flight must stay in flight)
        __builtin_amdgcn_sched_barrier(0);
        request_v(blk + 3, Vf);
        request_k(blk + 5, Kf);
        __builtin_amdgcn_sched_barrier(0);
    };
    auto share_tile = [&](auto maymask_tag, int jt, int nlive, half_t* K0, half_t* K1, half_t* K2, half_t* K3, half_t* V0, half_t* V1,
                          half_t* V3) __attribute__((always_inline)) {
        const int kv0 = kfirst + jt * KSTEP, g0 = grp * SR * D;
        auto none1 = [&](int) __attribute__((always_inline)) {};
        step(needs_mask(kv0 + 32), maymask_tag, std::true_type{}, sA, sB, V0 + g0, K1 + g0, K2 + g0, kv0 + 32,
             [&]() __attribute__((always_inline)) { share_handover(2 * jt, K1, V3); }, none1);
        more = jt + 1 < nlive;
        step(needs_mask(kv0 + KSTEP), maymask_tag, std::true_type{}, sB, sA, V1 + g0, K2 + g0, K3 + g0, kv0 + KSTEP,
             [&]() __attribute__((always_inline)) { share_handover(2 * jt + 1, K2, V0); }, none1);
    };
    // Under a causal mask the waves of a workgroup see different numbers of tiles: a wave computes the tiles that
    // hold a key visible to one of its queries, and for the rest only keeps up the staging it shares with the
    // others (its part of every refill, and the barrier), leaving its SIMD to the wave that still computes.
    int nlive = ntiles;
    if (a.causal) nlive = max(0, min(ntiles, (min(wq0 + 31, a.Sq - 1) + off) / BN + 1 - share * share_tiles));
    const int nloop = SPLIT ? (ntiles + 1) >> 1 : ntiles;
    if constexpr (SPLIT) nlive = (nlive - grp + 1) >> 1;           // (nlive = 0, grp = 1: 0)
    if (wq0 >= a.Sq) nlive = 0;             // no query of its own: the ragged end of a tile, or the middle tile of an odd count
    // The leading tiles whose blocks (and the first block of the tile after) lie wholly inside the keys and, under a
    // causal mask, before this wave's first query: a loop of their own without the mask test.  needs_mask is monotone
    // in the key index, so they are the tiles jt with 64 jt + 96 <= Skv and 64 jt + 95 <= wb; taken in pairs (the
    // stages alternate), the rest goes through the general loop.
    int n_plain = max(0, a.Skv - 32 - kfirst) / KSTEP;
    if (a.causal) n_plain = min(n_plain, max(0, wb - 31 - kfirst) / KSTEP);
    n_plain = min(n_plain, nlive) & ~1;
    if constexpr (SHARE) {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(0xc07f);     // lgkmcnt(0): K block 0 has been read ...
        __builtin_amdgcn_s_barrier();           // ... by everyone
        __builtin_amdgcn_sched_barrier(0);
        request_k(4, Ks0_);
        __builtin_amdgcn_sched_barrier(0);
        for (int jt = 0; jt < n_plain; jt += 2) {
            share_tile(std::false_type{}, jt, nlive, Ks0_, Ks1_, Ks2_, Ks3_, Vs0_, Vs1_, Vs3_);
            share_tile(std::false_type{}, jt + 1, nlive, Ks2_, Ks3_, Ks0_, Ks1_, Vs2_, Vs3_, Vs1_);
        }
        for (int jt = n_plain; jt < nlive; jt += 2) {
            share_tile(std::true_type{}, jt, nlive, Ks0_, Ks1_, Ks2_, Ks3_, Vs0_, Vs1_, Vs3_);
            if (jt + 1 < nlive) share_tile(std::true_type{}, jt + 1, nlive, Ks2_, Ks3_, Ks0_, Ks1_, Vs2_, Vs3_, Vs1_);
        }
        for (int jt = nlive; jt < nloop; ++jt) {
            share_handover(2 * jt, (jt & 1) ? Ks3_ : Ks1_, (jt & 1) ? Vs1_ : Vs3_);
            share_handover(2 * jt + 1, (jt & 1) ? Ks0_ : Ks2_, (jt & 1) ? Vs2_ : Vs0_);
        }
    } else {
        for (int jt = 0; jt < n_plain; jt += 2) {
            tile(std::false_type{}, jt, Ks0, Ks1, Vs0, Vs1);
            tile(std::false_type{}, jt + 1, Ks1, Ks0, Vs1, Vs0);
        }
        for (int jt = n_plain; jt < nlive; jt += 2) {
            tile(std::true_type{}, jt, Ks0, Ks1, Vs0, Vs1);
            if (jt + 1 < nlive) tile(std::true_type{}, jt + 1, Ks1, Ks0, Vs1, Vs0);
        }
        for (int jt = nlive; jt < nloop; ++jt) {
            half_t* Kc = (jt & 1) ? Ks1 : Ks0;
            half_t* Vn = (jt & 1) ? Vs0 : Vs1;
            __builtin_amdgcn_s_waitcnt(0x0f70);
            __syncthreads();
            if (jt + 2 < nloop) TRN_FETCH_K(jt + 2, Kc);
            if (jt + 1 < nloop) TRN_FETCH_V(jt + 1, Vn);
        }
    }
#undef TRN_FETCH_K
#undef TRN_FETCH_V

    // ---- epilogue: normalise; transpose this wave's 32 x D tile through LDS so that the stores are whole
    // 16-byte-per-lane row segments; LSEs ----
    float inv[2];
    float l[2];
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) { l[qb] = lacc[qb][0]; inv[qb] = 1.0f / l[qb]; }
    __builtin_amdgcn_s_waitcnt(0x0f70);                // this wave's last refills (past the end, unread) have landed ...
    __syncthreads();                                   // ... and everyone's; every wave is done with the K/V stages
    if constexpr (SPLIT) {
        // The groups hold partial results of the same queries.  Waves w and w + 4 (of two tiles, w and w ^ 6) exchange (m, l) and
        // halves of O^T lane by lane: group 0 finishes the first D/2 columns, group 1 the others.  A wave that took no tile, or a
        // query that saw no key of its group, has zero sums and weighs nothing.
        const int other = wave ^ (even ? 6 : 4);
        constexpr int kStat = D == 128 ? 5120 : 2560;   // (floats) the row statistics lie behind the transposing regions
        float* stat = SHARE ? reinterpret_cast<float*>(Ks2_) : reinterpret_cast<float*>(Ks1_) + kStat;   // [8 waves][2 query blocks][16 queries] {m, l}
#pragma unroll
        for (int qb = 0; qb < 2; ++qb) {
            if (nlive == 0 || fresh[qb]) m[qb] = -INFINITY;
            if (g4 == 0) {
                stat[((wave * 2 + qb) * 16 + n) * 2] = m[qb];
                stat[((wave * 2 + qb) * 16 + n) * 2 + 1] = l[qb];
            }
        }
        constexpr int NH = NOP / 2;
        float4_t* mine = reinterpret_cast<float4_t*>(wave < 4 ? Ks0_ : Vs0_) + (wave & 3) * NH * 2 * 64;
        const float4_t* theirs = reinterpret_cast<const float4_t*>(wave < 4 ? Vs0_ : Ks0_) + (other & 3) * NH * 2 * 64;
        if constexpr (SHARE) {          // (a stage of the ring holds two waves' halves)
            half_t *const ka_ = wave & 2 ? Ks1_ : Ks0_, *const va_ = wave & 2 ? Vs1_ : Vs0_;
            mine = reinterpret_cast<float4_t*>(wave < 4 ? ka_ : va_) + (wave & 1) * NH * 2 * 64;
            theirs = reinterpret_cast<const float4_t*>(wave < 4 ? va_ : ka_) + (wave & 1) * NH * 2 * 64;
        }
#pragma unroll
        for (int i = 0; i < NH; ++i)
#pragma unroll
            for (int qb = 0; qb < 2; ++qb) mine[(i * 2 + qb) * 64 + lane] = grp == 0 ? oacc[NH + i][qb] : oacc[i][qb];
        __syncthreads();
        float wo[2], wt[2];
#pragma unroll
        for (int qb = 0; qb < 2; ++qb) {
            const float mt = stat[((other * 2 + qb) * 16 + n) * 2], lt = stat[((other * 2 + qb) * 16 + n) * 2 + 1];
            float ms = fmaxf(m[qb], mt);                  // (finite: every query sees a key -- but not of every share)
            if (SHARE && ms == -INFINITY) ms = 0.f;
            wo[qb] = fast_exp2(m[qb] - ms); wt[qb] = fast_exp2(mt - ms);
            l[qb] = l[qb] * wo[qb] + lt * wt[qb];
            m[qb] = ms;
            inv[qb] = 1.0f / l[qb];
        }
#pragma unroll
        for (int i = 0; i < NH; ++i)
#pragma unroll
            for (int qb = 0; qb < 2; ++qb) {
                const float4_t own = grp == 0 ? oacc[i][qb] : oacc[NH + i][qb];
                oacc[i][qb] = own * wo[qb] + theirs[(i * 2 + qb) * 64 + lane] * wt[qb];
            }
        if constexpr (SHARE) {
            // this share's {O unnormalised, m, l} per query, fp32: rows of D floats, then the pairs of all rows
            // (3 MB and more of them past the caches, as far as the L2s would be written back at the end of the launch: with the merge,
            // us, through / past, K and V out of the caches: 32 heads of 128: 100 queries on 4.1 k keys (13 MB) 26.8 / 25.4, 128 on 3.2 k 28.0 /
            // 26.1, 40 on 3.1 k (5.3) 19.8 / 19.1; 16 of 64: 100 on 4.1 k 16.9 / 15.8, 60 on 4.3 k (4.1) 14.85 / 14.55, 50 on 4.2 k (3.4) 14.41 /
            // 14.31, 40 on 4.1 k (2.7) 14.34 / 14.56; 8 of 128: 40 on 3.1 k (2.7) 15.64 / 15.94; 71 of 64: 64 on 6 k (3.6) 29.9 / 29.9, 40 on 6 k (2.2)
            // 29.1 / 29.4)
            const int64_t rows = (int64_t)a.heads.all.d * a.n_split * a.Sq, row0 = ((int64_t)(b * a.Hq + head) * a.n_split + share) * a.Sq;
            const int past = rows * D * 4 >= (int64_t)3 << 20 ? 1 : 0;
#pragma unroll
            for (int qb = 0; qb < 2; ++qb) {
                if (qrow[qb] >= a.Sq) continue;
                float* po = a.ws + (row0 + qrow[qb]) * D + grp * (D / 2) + 4 * g4;
#pragma unroll
                for (int i = 0; i < NH; ++i) store_out(po + 16 * i, oacc[i][qb], past);
                if (g4 == 0 && grp == 0) *reinterpret_cast<float2_t*>(a.ws + rows * D + (row0 + qrow[qb]) * 2) = float2_t{l[qb] > 0.f ? m[qb] : -INFINITY, l[qb]};
            }
            return;
        }
        constexpr int DP = D / 2, OP = DP + 4, LPRW = DP / 8, RPS = 64 / LPRW;
        half_t* ot = (wave < 4 ? Vs1_ : Ks1_) + (wave & 3) * 32 * OP;
        static_assert(4 * 32 * OP * 2 <= kStat * 4 && kStat * 4 + 2048 <= 2 * BN * D * 2, "the stage holds both");
        const int orow = lane / LPRW, ocol = (lane % LPRW) * 8;
        half_t* ob = a.o + b * a.ob + head * a.oh + grp * DP;
#pragma unroll
        for (int dbl = 0; dbl < NH; ++dbl)
#pragma unroll
            for (int qb = 0; qb < 2; ++qb) {
                half4_t ov;
#pragma unroll
                for (int e = 0; e < 4; ++e) ov[e] = (half_t)(oacc[dbl][qb][e] * inv[qb]);
                *reinterpret_cast<half4_t*>(&ot[(16 * qb + n) * OP + dbl * 16 + 4 * g4]) = ov;
            }
#pragma unroll
        for (int jj = 0; jj < 32 / RPS; ++jj) {
            const int r = jj * RPS + orow;
            const uint2_t lo = *reinterpret_cast<const uint2_t*>(&ot[r * OP + ocol]);
            const uint2_t hi = *reinterpret_cast<const uint2_t*>(&ot[r * OP + ocol + 4]);
            if (wq0 + r < a.Sq)
                store_out(ob + (int64_t)(wq0 + r) * a.os + ocol, uint4_t{lo.x, lo.y, hi.x, hi.y}, a.o_nt);
        }
        if (grp == 1) return;               // (the LSEs are written once)
    } else {
        // two passes of D/2 columns each, so that NW waves' staging regions fit in the four stage arrays
        constexpr int DP = D / 2, OP = DP + 4;         // row pitch in halfs
        constexpr int LPRW = DP / 8, RPS = 64 / LPRW;  // lanes per output row segment, rows per store instruction
        static_assert(32 * OP * 2 <= BN * D * 2 / (NW / 4), "staging region too large");
        half_t* arr = (wave / (NW / 4)) == 0 ? Ks0 : (wave / (NW / 4)) == 1 ? Ks1 : (wave / (NW / 4)) == 2 ? Vs0 : Vs1;
        half_t* ot = arr + (wave % (NW / 4)) * (BN * D / (NW / 4));
        const int orow = lane / LPRW, ocol = (lane % LPRW) * 8;
        half_t* ob = a.o + b * a.ob + head * a.oh;
#pragma unroll
        for (int pass = 0; pass < 2; ++pass) {
#pragma unroll
            for (int dbl = 0; dbl < NOP / 2; ++dbl)
#pragma unroll
                for (int qb = 0; qb < 2; ++qb) {
                    half4_t ov;
#pragma unroll
                    for (int e = 0; e < 4; ++e) ov[e] = (half_t)(oacc[pass * (NOP / 2) + dbl][qb][e] * inv[qb]);
                    *reinterpret_cast<half4_t*>(&ot[(16 * qb + n) * OP + dbl * 16 + 4 * g4]) = ov;
                }
            // (LDS operations of one wave execute in order: no wait needed between its own writes and reads)
#pragma unroll
            for (int jj = 0; jj < 32 / RPS; ++jj) {
                const int r = jj * RPS + orow;
                const uint2_t lo = *reinterpret_cast<const uint2_t*>(&ot[r * OP + ocol]);
                const uint2_t hi = *reinterpret_cast<const uint2_t*>(&ot[r * OP + ocol + 4]);
                if (wq0 + r < a.Sq)
                    store_out(ob + (int64_t)(wq0 + r) * a.os + pass * DP + ocol, uint4_t{lo.x, lo.y, hi.x, hi.y}, a.o_nt);
            }
        }
    }
    if (g4 == 0 && a.lse) {
#pragma unroll
        for (int qb = 0; qb < 2; ++qb)
            if (qrow[qb] < a.Sq) a.lse[((int64_t)b * a.Hq + head) * a.Sq + qrow[qb]] = (m[qb] + fast_log2(l[qb])) * kLn2;
    }
}
#endif

template <int D, int NW, bool PAIRED>
__global__ __launch_bounds__(NW * 64, NW == 8 ? 1 : 2) void attn_fwd16_kernel(const AttnArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
    attn_fwd16_body<D, NW, PAIRED ? kPaired : kPlain>(a);
#endif
}

template <int D>
__global__ __launch_bounds__(512, 1) void attn_fwd16_split_kernel(const AttnArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
    attn_fwd16_body<D, 8, kSplit>(a);
#endif
}

template <int D, int NW, int MODE>
__global__ __launch_bounds__(NW * 64, NW == 8 ? 1 : 2) void attn_fwd16_given_kernel(const AttnArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
    // (KeyFormer's sums of a head's workgroups ride along behind the attention's own workgroups.  Whole calls, us, a launch of their own / so: 71 heads of
    // 64, 400 keys 23.1 / 20.8, 777 fp16 41.3 / 39.9, 32 of 128, 1000 fp16 43.2 / 41.3, 2 x 16 of 64, 1000 31.7 / 29.3)
    if ((int)blockIdx.x >= a.n_main) {
        add_slots(a.sums, (int64_t)((int)blockIdx.x - a.n_main) * (NW * 64) + threadIdx.x);
        return;
    }
    attn_fwd16_body<D, NW, MODE, true>(a);
#endif
}

template <int D>
__global__ __launch_bounds__(512, 1) void attn_fwd16_share_kernel(const AttnArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
    attn_fwd16_body<D, 8, kShare>(a);
#endif
}

constexpr int kMaxShares = 16;

// The shares' results of one query per wave: D / 64 columns per lane, the shares in order.  Two memory latencies and the
// launch, 4 - 5 us (with the shares' maxima and sums read by every lane in a loop of its own, 5 - 8).
template <int D>
__global__ __launch_bounds__(256) void attn_merge_shares_kernel(const AttnArgs a) {
    const int lane = threadIdx.x & 63;
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6), n_rows = (int64_t)a.B * a.Hq * a.Sq;
    if (row >= n_rows) return;
    const int64_t bh = row / a.Sq, qr = row % a.Sq, b = bh / a.Hq, head = bh % a.Hq;
    const float* parts = a.ws + (bh * a.n_split * a.Sq + qr) * D;                            // share s: + s * Sq * D
    const float* st = a.ws + n_rows * a.n_split * D + (bh * a.n_split * a.Sq + qr) * 2;      // share s: + s * Sq * 2
    constexpr int C = D / 64, BATCH = 8;
    // lane s holds share s's {m, l}; the first rows are requested before they are waited for
    const float2_t ml = *reinterpret_cast<const float2_t*>(st + (int64_t)min(lane, a.n_split - 1) * a.Sq * 2);
    float r[BATCH][C];
    auto fetch = [&](int s0) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < BATCH; ++u)
#pragma unroll
            for (int i = 0; i < C; ++i) r[u][i] = parts[(int64_t)min(s0 + u, a.n_split - 1) * a.Sq * D + lane * C + i];
    };
    fetch(0);
    float m = ml.x;
#pragma unroll
    for (int k = 1; k < kMaxShares; k <<= 1) m = fmaxf(m, __shfl_xor(m, k, 64));
    const float w = lane < a.n_split ? fast_exp2(ml.x - m) : 0.f;       // (lanes past the shares repeat the last one's m)
    float l = lane < kMaxShares ? w * ml.y : 0.f;
#pragma unroll
    for (int k = 1; k < kMaxShares; k <<= 1) l += __shfl_xor(l, k, 64);
    l = __shfl(l, 0, 64); m = __shfl(m, 0, 64);
    float o[C] = {};
    for (int s0 = 0; s0 < a.n_split; s0 += BATCH) {
#pragma unroll
        for (int u = 0; u < BATCH; ++u) {
            const float wu = s0 + u < a.n_split ? __shfl(w, s0 + u, 64) : 0.f;
#pragma unroll
            for (int i = 0; i < C; ++i) o[i] = __builtin_fmaf(r[u][i], wu, o[i]);
        }
        if (s0 + BATCH < a.n_split) fetch(s0 + BATCH);
    }
    half_t* orow = a.o + b * a.ob + head * a.oh + qr * a.os + lane * C;
#pragma unroll
    for (int i = 0; i < C; ++i) orow[i] = (half_t)(o[i] / l);
    if (lane == 0 && a.lse) a.lse[row] = (m + fast_log2(l)) * kLn2;
}

// Key shares of the query tiles of 128, one workgroup per CU in all (0: the keys are not shared out).  The other forms are
// tiles of 32 queries with all the keys each (attn_decode.hip: every tile reads K and V again, twice or more with its column
// shares) and workgroups of 128 queries (a CU per tile).  Shares read the cache once, at some 8 us + 6 TB/s, and pay about
// 5 us for the merge: not on short caches.  us without / with shares (both launches): 32 heads of 128: 100 queries on 2.6 k
// keys 20.7 / 20.8, 128 on 2.8 k 21.1 / 22.7, 128 on 3.1 k 25.6 / 23.9, 40 on 2.7 k 19.3 / 18.1, 3 k 23.4 / 19.5, 100 on 4.1 k
// 32.1 / 24.1, 128 on 8.1 k 56.8 / 41, 50 on 16 k 98 / 55, 300 on 4.3 k 61.5 / 48; 8 heads of 128: 100 on 2.6 k 16.2 / 16.0, 40
// on 3 k 17.6 / 15.5, 500 on 3.5 k 25.6 / 23.0, 128 on 16 k 73 / 28; 16 heads of 64: 100 on 2.1 k 10.5 / 13.5, 3.1 k 13.9 / 13.4,
// 40 on 4 k 15.4 / 13.6, 128 on 9.1 k 30 / 18; 71 heads of 64: 64 on 3.1 k 16.2 / 20.2, 4.1 k 25.1 / 23.0, 40 on 6 k 33.8 / 29.3,
// and, with more than 256 tiles of 32 queries, 100 on 1.3 k 16.7 / 16.4, 1.6 k 18.8 / 16.9, 2.6 k 29.0 / 19.9, 128 on 16 k 137 / 65.
static int key_shares(int64_t bh, int seq_q, int seq_kv, int head_dim) {
    const int64_t tiles = ((int64_t)seq_q + 127) / 128 * bh, tiles32 = ((int64_t)seq_q + 31) / 32 * bh;
    if (seq_q <= 32 || tiles > 128 || seq_kv < (head_dim == 128 ? 3072 : tiles32 > 256 ? 2560 : 4096)) return 0;
    return (int)min((int64_t)kMaxShares, 256 / tiles);
}

// The decode kernel keeps the arrival counters of its key splits (128 heads at most) at the head of a workspace and relies on
// finding them zero: the shares stay behind them, so that one zero-filled workspace serves both kinds of call.
constexpr int64_t kCounterBytes = 512;

int64_t attn_share_workspace_bytes(int batch, int n_q_heads, int seq_q, int seq_kv, int head_dim) {
    const int64_t bh = (int64_t)batch * n_q_heads;
    const int shares = key_shares(bh, seq_q, seq_kv, head_dim);
    return shares == 0 ? 0 : kCounterBytes + bh * shares * seq_q * (head_dim + 2) * 4;
}

template <int D>
static hipError_t launch_shares(AttnArgs a, hipStream_t s) {
    a.ws += kCounterBytes / sizeof(float);
    a.n_qtiles = (a.Sq + 127) / 128;
    a.n_split = key_shares((int64_t)a.B * a.Hq, a.Sq, a.Skv, D);
    hipLaunchKernelGGL((attn_fwd16_share_kernel<D>), dim3((unsigned)(a.n_qtiles * a.B * a.Hq * a.n_split)), dim3(512), 0, s, a);
    if (const hipError_t e = hipGetLastError(); e != hipSuccess) return e;
    hipLaunchKernelGGL((attn_merge_shares_kernel<D>), dim3((unsigned)(((int64_t)a.B * a.Hq * a.Sq + 3) / 4)), dim3(256), 0, s, a);
    return hipGetLastError();
}
hipError_t launch_attn_shares(const AttnArgs& a, int head_dim, hipStream_t s) {
    return head_dim == 128 ? launch_shares<128>(a, s) : launch_shares<64>(a, s);
}

// How many heads of a KV head a narrow workgroup takes, as a power of two: 2^pack heads times 4 / 2^pack blocks of 32 queries instead of
// four blocks of one head.  The tiles are then shorter by as much, their waves see the same keys, and a last tile of few queries, whose
// walk is the longest, is a quarter as large.  Where workgroups come in more than one round, up to 2048 keys; not where one round holds them, since
// the longest tile then has four waves with a full walk each.  us, one head / two / four:
//   32 heads of 128 on 8: 4 x 520 tokens 20.9 / 19.0 / 16.9, 4 x 777 30.8 / 30.2 / 29.8, 3 x 777 26.4 / 24.3 / 24.4, 8 x 400 23.5 / 21.8 / 21.5, 2 x 1600
//     49.5 / 46.8 / 46.8, 2250 47.4 / 46.9 / 47.2; 8 x 8 on 2, 1300 36.5 / 33.6 / 33.8; left out: 2 x 700 (384 workgroups of one head) 15.9 / 16.4 / 16.4, 8 x 250
//     (512) 11.8 / 11.9 / 11.9, 8 x 8 on 2, 777 (448) 17.8 / 18.1 / 18.6, 4 x 8 on 2, 2600 55.9 / 57.0 / 56.8
//   71 of 64 on one: 700 (426) 11.7 / 11.2 / 11.2, 2 x 300 (426) 9.0 / 7.8 / 7.9, 8 x 130 11.8 / 9.7 / 7.9, 4 x 400 16.2 / 13.8 / 13.5, 1600 30.7 / 29.4 / 29.2, 3600
//     121 / 118 / 117; left out: 520 (355) 9.4 / 9.3 / 9.5, 300 (213) 7.1 / 7.2 / 7.5, 3 x 223 (426)
//     7.7 against 7.9 of four (4 x 256 9.5 and 8.45)
// (heads that do not fill the last workgroup leave its waves idle: a sixteenth of them at most, and hardly any of short prompts without a ragged
// last tile to gain from: 12 groups of 21 heads of 64, 383 tokens, one head / two 11.8 / 12.7, 28 of 35 of 128, 255 50.3 / 54.7 of four)
static int packed_heads(int batch, int n_kv_heads, int group, int seq_q, int seq_kv, int head_dim, bool causal) {
    const int64_t narrow = ((int64_t)seq_q + 127) / 128 * batch * n_kv_heads * group;
    if (!causal || seq_q != seq_kv || !(head_dim == 128 ? narrow > 512 && seq_kv <= 2048 : narrow >= (seq_q > 256 ? 400 : 512))) return 0;
    int p = 2;
    const int64_t part = seq_q <= 384 && (seq_q - 1) % 128 >= 96 ? 50 : 16;
    while (p > 0 && (((int64_t)(group - 1) >> p) + 1) * part << p > (int64_t)group * (part + 1)) --p;
    return p;
}

// Whether a workgroup with split keys takes two tiles of 64 queries from the two ends of a causal problem instead of 128 consecutive
// ones: as many workgroups, all of the same work.  Where they run all at once (each needs a CU), the longest of the others sets the time.
// us, one tile / two: 8 heads of 128: 1300 keys 21.1 / 18.8, 2048 28.8 / 24.4, 3000 39.3 / 32.8, 4096 50.7 / 43.6; 16: 1500 23.5 / 21.0, 2000
// 29.0 / 26.3; 24: 1200 21.5 / 19.7; 16 heads of 64: 1300 14.1 / 12.6, 2048 19.1 / 16.7, and against narrow workgroups (Attn16Shape) 600
// 9.6 / 9.4, 777 11.1 / 10.2, 32 heads: 640 9.8 / 9.6, 900 12.5 / 11.1, 1020 13.8 / 11.7, but 520 9.0 / 9.1; 16 heads, 3000 keys (384 workgroups) 27.3 / 34.6.
static bool split_in_two(int64_t batch, int64_t n_q_heads, int64_t seq_q, int64_t seq_kv, bool causal) {
    return causal && seq_q == seq_kv && (seq_q + 127) / 128 * batch * n_q_heads <= 256;
}

template <int D, int NW, int MODE, bool GIVEN>
static hipError_t launch16(AttnArgs a, hipStream_t s) {
    a.even = MODE == kSplit && split_in_two(a.B, a.Hq, a.Sq, a.Skv, a.causal != 0);
    a.pack = MODE == kPlain && NW == 4 ? packed_heads(a.B, a.Hkv, a.heads.G, a.Sq, a.Skv, D, a.causal != 0) : 0;
    if (a.pack) a.heads.all = Div((int64_t)a.B * a.Hkv * (((a.heads.G - 1) >> a.pack) + 1));
    const int rows = MODE == kPlain ? 32 * NW >> a.pack : a.even ? 64 : 128;
    a.n_qtiles = (int)(((int64_t)a.Sq + rows - 1) / rows);
    const int64_t grid = (int64_t)(MODE == kPaired || a.even ? (a.n_qtiles + 1) / 2 : a.n_qtiles) * a.heads.all.d;
    const int64_t more = GIVEN && a.sums.n_slots > 0 ? (a.sums.n + NW * 64 - 1) / (NW * 64) : 0;
    if (grid + more > 0x7fffffffLL) return hipErrorInvalidValue;
    a.n_main = (int)grid;
    if constexpr (GIVEN) hipLaunchKernelGGL((attn_fwd16_given_kernel<D, NW, MODE>), dim3((unsigned)(grid + more)), dim3(NW * 64), 0, s, a);
    else if constexpr (MODE == kSplit) hipLaunchKernelGGL((attn_fwd16_split_kernel<D>), dim3((unsigned)grid), dim3(NW * 64), 0, s, a);
    else hipLaunchKernelGGL((attn_fwd16_kernel<D, NW, MODE == kPaired>), dim3((unsigned)grid), dim3(NW * 64), 0, s, a);
    return hipGetLastError();
}

// Workgroup shape by problem size (the figures are us, llama heads = 32 query / 8 KV heads of 128; W counts narrow
// workgroups).  All four shapes cost the same per wave and 64-key tile, about 0.9 us; what differs is how many waves a
// CU holds and which of them ends last.
//  Narrow  128 queries, four waves, two workgroups per CU: the general case.
//  Split   the same 128 queries by eight waves, which halves the walk over the keys and adds a merge (2 - 3 us).  Pays
//          when every workgroup has a CU to itself anyway and the walk is long: W <= 256 and 1100 keys or more
//          (8 heads of 128, 3000 tokens: 42.2 against 46.8; 16 heads of 64, 2000: 21.2 against 23.3; 250 queries on
//          3250 keys: 46.0 against 51.0; but 1000 tokens, 16 heads of 128: 20.5 against 20.7, 600: 15.6 against 14.9).
//          A causal triangle's short tiles leave room for a few more: W <= 320 (16 heads of 128, 2500: 40.1 against
//          41.7 paired; at W = 416: 35.1 against 31.9).  Up to 256 a causal problem's workgroups take two short tiles each
//          (split_in_two), which with head_dim 64 pays from 600 keys on.
//  Paired  a causal problem whose narrow workgroups are all resident at once: the longest tile sets the time, twice the
//          mean, so each workgroup takes two tiles from opposite ends.  Such workgroups are half as many and each needs
//          a CU of its own: 192 to 256 of them (2048 tokens, llama heads: 40.5 against 44.4 narrow; at 288 workgroups,
//          71 heads of 64 and 777 tokens: 20.2 against 13.8), and tiles enough for an imbalance to matter (at 12 tiles
//          30.3 against 31.4, at 11 28.3 against 27.1).
//  Wide    256 queries per K/V stage (head_dim 128 only; with 64 it loses 10 - 20 % at every size): fewer LDS fills and
//          a few % less energy, where the chip is full and the power limit sets the pace.  Unmasked, from one workgroup
//          per CU; causal, where tiles of different lengths must even out over rounds, from 384 workgroups of at least
//          four tiles per head if the last tile is nearly full (llama heads, 4096: 121 against 133.5; 3500: 92.9 against
//          101.9; two of 1700: 54 against 58.3; but eight of 512, two tiles: 34.3 against 30.3, and eight of 1300, whose
//          sixth tile holds 20 rows: 156 against 140).
Attn16Shape attn_fwd16_shape(int batch, int n_q_heads, int seq_q, int seq_kv, int head_dim, bool causal) {
    const int64_t bh = (int64_t)batch * n_q_heads;
    const int64_t n128 = ((int64_t)seq_q + 127) / 128, W = n128 * bh;
    if (seq_kv >= 1100 && (W <= 256 || (causal && seq_kv == seq_q && W <= 320))) return Attn16Shape::Split;
    if (head_dim == 64 && seq_kv >= 600 && split_in_two(batch, n_q_heads, seq_q, seq_kv, causal)) return Attn16Shape::Split;
    const int64_t pairs = ((n128 + 1) / 2) * bh;
    if (causal && W <= 512 && pairs >= 192 && pairs <= 256 && n128 >= 12) return Attn16Shape::Paired;
    const int64_t n256 = ((int64_t)seq_q + 255) / 256;
    const bool wide = causal ? n256 * bh >= 384 && n256 >= 4 && n256 * 256 * 16 <= (int64_t)seq_q * 17 : n256 * bh >= 256;
    return head_dim == 128 && wide ? Attn16Shape::Wide : Attn16Shape::Narrow;
}

template <bool GIVEN>
static hipError_t launch_shape(const AttnArgs& a, bool d128, Attn16Shape shape, hipStream_t s) {
    switch (shape) {
        case Attn16Shape::Paired: return d128 ? launch16<128, 8, kPaired, GIVEN>(a, s) : launch16<64, 8, kPaired, GIVEN>(a, s);
        case Attn16Shape::Split:  return d128 ? launch16<128, 8, kSplit, GIVEN>(a, s) : launch16<64, 8, kSplit, GIVEN>(a, s);
        case Attn16Shape::Wide:   return launch16<128, 8, kPlain, GIVEN>(a, s);             // (head_dim 128 only)
        default:                  return d128 ? launch16<128, 4, kPlain, GIVEN>(a, s) : launch16<64, 4, kPlain, GIVEN>(a, s);
    }
}
hipError_t launch_attn_fwd16(const AttnArgs& a, int head_dim, Attn16Shape shape, bool given_q, hipStream_t s) {
    return given_q ? launch_shape<true>(a, head_dim == 128, shape, s) : launch_shape<false>(a, head_dim == 128, shape, s);
}

const char* attn_fwd16_kernel_name(int head_dim, Attn16Shape shape) {
    if (shape == Attn16Shape::Split) return head_dim == 128 ? "trn::attn_fwd16_split_kernel<128>" : "trn::attn_fwd16_split_kernel<64>";
    if (shape == Attn16Shape::Paired) return head_dim == 128 ? "trn::attn_fwd16_kernel<128, 8, true>" : "trn::attn_fwd16_kernel<64, 8, true>";
    if (shape == Attn16Shape::Wide) return "trn::attn_fwd16_kernel<128, 8, false>";
    return head_dim == 128 ? "trn::attn_fwd16_kernel<128, 4, false>" : "trn::attn_fwd16_kernel<64, 4, false>";
}

}  // namespace trn
