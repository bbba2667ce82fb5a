// KeyFormer's perturbed row normalisers and key scores in one pass over the noise:
//
//     lse_i = log sum_j exp(z_ij),   out_j = sum_i exp(z_ij - lse_i),   z = (scale * Q K^T + noise) / tau
//
// A column sum needs the finished row normalisers, so that two passes -- the forward's, row by row, and the statistics', column
// by column -- read all of the noise twice, at the rate of HBM both times (the last-level cache returns lines no faster than
// HBM: a 128 MB buffer read over and over 7.0 - 7.4 TB/s, 2 GB 6.3 - 7.1).  Here a workgroup takes 32 queries at a time and keeps their
// exponentials in registers, 32 x 2048 of them in fp32 -- half of a CU's register file --, until the rows are summed up; the
// scores then follow without another look at the noise.  Only what a row has beyond 2048 keys is read, and multiplied, again.
// The attention itself, which does not depend on the noise, runs on the kernels of attn_fwd16.hip with the queries as given.
//
// Eight waves take a strip's 32-key blocks in turn, each through a private part of LDS (K one block ahead, noise two), so that
// the walk has no barrier.  S[query][key], a lane one key and 16 of the 32 queries: the scores' sums over the queries are then
// sums within a lane, the blocks of a wave are the same columns in every strip, and a workgroup adds them up in LDS without
// atomics; the launch of the attention behind this one adds the workgroups of a head in a fixed order.  Results repeat bit for bit.
//
// What bounds it: a wave's block is a chain -- K and noise out of LDS, eight MFMAs that wait for each other, the exponentials --
// that two waves a SIMD overlap only in part, and 32 to 64 KB of noise in flight a CU.  71 heads of 64, 1536 keys, fp32: 79 us for
// 0.37 GB (4.7 TB/s; 59 with the noise in the caches, 51 without its and K's requests at all); 32 heads of 128, 2048: 83 us, where
// the forward's noise and the statistics took 121 beside the attention's 42.
//
// All requests are global -> LDS loads issued as inline assembly and counted by hand: a wave's requests run ahead over the end
// of a strip into the next, and the compiler, which cannot see which of them a read depends on, would wait for all.
#include "attn.h"

namespace trn {

struct StripArgs {
    const half_t* q; const half_t* k; const void* noise; float* lse; float* out; float* part;
    int B, Hq, Hkv, S, n_strips, n_slots, missing;
    HeadMap heads;
    int64_t qb, qh, qs, kb, kh, ks, nb, nh, ns;
    float c2, c3;      // scale*log2(e)/tau, log2(e)/tau
    int s16;
};

[[maybe_unused]] constexpr int kHeldBlocks = 8;      // of 32 keys, per wave
// keys whose column sums fit beside the stages, of 8 waves a CU in one workgroup or two
constexpr int strip_keys(int waves, int head_dim) { return waves == 8 ? 4864 : head_dim == 128 ? 1664 : 5120; }

#if defined(__HIP_DEVICE_COMPILE__)
// Four of a wave's global -> LDS loads of BYTES a lane, LSTEP bytes of LDS and `step` bytes of memory from each to the next:
// lane l's land at lds + 4 l (16 l), offsets past the range as zeros.  lds and so end up where a fifth would go.
// (m0, which both functions write, is a reserved register that a clobber list does not take: this kernel has no other user of it --
// no global -> LDS load by a builtin, no message, no indexed register.  so is written before the last inputs are read.)
template <int BYTES, bool NT, int LSTEP>
__device__ __forceinline__ void request4(uint4_t rs, uint32_t& lds, int vo0, int vo1, int vo2, int vo3, int& so, int step) {
#define TRN_NEXT "s_add_u32 m0, m0, %8\n\ts_add_u32 %0, %0, %7\n\t"
#define TRN_REQ(op_, mod_)                                                                                                      \
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\t" op_ " %2, %6, %0 offen " mod_ "\n\t" TRN_NEXT op_ " %3, %6, %0 offen " mod_ "\n\t" TRN_NEXT    \
                 op_ " %4, %6, %0 offen " mod_ "\n\t" TRN_NEXT op_ " %5, %6, %0 offen " mod_ "\n\ts_add_u32 %0, %0, %7"         \
                 : "+&s"(so) : "s"(lds), "v"(vo0), "v"(vo1), "v"(vo2), "v"(vo3), "s"(rs), "s"(step), "n"(LSTEP) : "memory", "scc")
    if constexpr (BYTES == 16) { if constexpr (NT) TRN_REQ("buffer_load_dwordx4", "nt lds"); else TRN_REQ("buffer_load_dwordx4", "lds"); }
    else if constexpr (BYTES == 4) TRN_REQ("buffer_load_dword", "lds");
    else TRN_REQ("buffer_load_ushort", "lds");
#undef TRN_REQ
#undef TRN_NEXT
    lds += 4 * LSTEP;
}
__device__ __forceinline__ void request1(uint4_t rs, uint32_t lds, int vo, int so) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" :: "s"(lds), "v"(vo), "s"(rs), "s"(so) : "memory");
}
template <int N> __device__ __forceinline__ void wait_requests() { asm volatile("s_waitcnt vmcnt(%0)" :: "n"(N) : "memory"); }
__device__ __forceinline__ void wait_lds() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }
__device__ __forceinline__ uint32_t lds_address(const void* p) { return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)p; }
__device__ __forceinline__ half8_t operand(uint32_t at) { return *(__attribute__((address_space(3))) const half8_t*)(uintptr_t)at; }
__device__ __forceinline__ uint4_t descriptor(const void* p, int64_t bytes) {
    const uint64_t u = reinterpret_cast<uint64_t>(p);
    return uint4_t{(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)u), (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(u >> 32)),
                   (uint32_t)__builtin_amdgcn_readfirstlane((int)bytes), 0x00020000u};
}

template <int CTRL> __device__ __forceinline__ float dpp(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xf, 0xf, true));
}
// The lane, where it is not worth a register over the walk.
__device__ __forceinline__ int lane_now() {
    int r;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(r));
    return r;
}
// f over the 32 lanes of each half, of 16 values a lane: lane l ends with that of value l % 16.  Each step hands half of the
// values to a lane that differs in one more bit of its number (ror 8, half mirror, two quad permutations) and keeps the others.
template <class F>
__device__ __forceinline__ float reduce_keys(const float (&v)[16], int lane, F f) {
    float a[8], b[4], c[2];
    const bool b3 = lane & 8, b2 = lane & 4, b1 = lane & 2, b0 = lane & 1;
#pragma unroll
    for (int i = 0; i < 8; ++i) a[i] = f(b3 ? v[i + 8] : v[i], dpp<0x128>(b3 ? v[i] : v[i + 8]));
#pragma unroll
    for (int i = 0; i < 4; ++i) b[i] = f(b2 ? a[i + 4] : a[i], dpp<0x141>(b2 ? a[i] : a[i + 4]));
#pragma unroll
    for (int i = 0; i < 2; ++i) c[i] = f(b1 ? b[i + 2] : b[i], dpp<0x4e>(b1 ? b[i] : b[i + 2]));
    float x = f(b0 ? c[1] : c[0], dpp<0xb1>(b0 ? c[0] : c[1])), y = x;
    asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(x), "+v"(y));
    return f(x, y);
}
#endif

// NB: bytes of noise a lane requests at a time: 16 fp32 rows on 16-byte addresses, 4 fp32, 2 fp16.
template <int D, int NB, bool NT, int NW>
__global__ __launch_bounds__(NW * 64, NW == 8 ? 1 : 2) void attn_noise_strips_kernel(const StripArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
    constexpr int NKS = D / 16, CPR = D / 8, RPI = 64 / CPR;
    constexpr int NK = 32 / RPI;                 // requests of a block's K
    constexpr int NN = NB == 16 ? 4 : 16;        // ... and of its noise
    constexpr int nsz = NB == 2 ? 2 : 4, NQW = 8 / NW, kKeys = strip_keys(NW, D);
    __shared__ __attribute__((aligned(1024))) half_t Ks[NW * 32 * D];
    __shared__ __attribute__((aligned(1024))) float Ns[NW * 2 * 1024];
    __shared__ __attribute__((aligned(1024))) half_t Qs[32 * D];
    __shared__ __attribute__((aligned(256))) float2_t St[NW * 32];       // a strip's row references and sums, by wave
    __shared__ __attribute__((aligned(256))) float Wr[NW * 32];          // a value per row: the references, or what one lane has for all
    __shared__ __attribute__((aligned(256))) float Cs[kKeys];                // the column sums

    const int tid = threadIdx.x, lane = tid & 63, c = lane & 31, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int slot = a.heads.all.of(blockIdx.x);
    int b, kvh, g;
    a.heads.find(blockIdx.x - slot * a.heads.all.d, b, kvh, g);
    const int head = kvh * a.heads.G + g;

    const uint4_t qrs = descriptor(a.q + b * a.qb + head * a.qh, ((int64_t)(a.S - 1) * a.qs + D) * 2);
    const uint4_t krs = descriptor(a.k + b * a.kb + kvh * a.kh, ((int64_t)(a.S - 1) * a.ks + D) * 2);
    const uint4_t nrs = descriptor(static_cast<const char*>(a.noise) + (b * a.nb + head * a.nh) * nsz, ((int64_t)(a.S - 1) * a.ns + a.S) * nsz);

    // ---- K and Q: RPI rows a request, the 16-byte chunks of a row swizzled by its number on their way in
    const int krow = lane / CPR;
    int kvo[D == 128 ? 4 : 2];                   // (the swizzle's part that differs from request to request)
#pragma unroll
    for (int p = 0; p < (D == 128 ? 4 : 2); ++p) kvo[p] = (int)(krow * a.ks * 2) + (((lane % CPR) ^ swz<D>(p * RPI + krow)) << 4);
    // ---- noise: row 8p + 4h + i of a block at 1024 p + 256 i + 128 h bytes, its keys in order: what a lane reads of row number r
    // of its 16 lies at 256 r + 4 lane
    const int nvo = NB == 16 ? (int)((4 * ((lane >> 3) & 1) + (lane >> 4)) * a.ns * 4) + 16 * (lane & 7) : (int)((4 * h * a.ns + c) * nsz);
    float* const nst = Ns + wave * 2 * 1024;
    const uint32_t klds = lds_address(Ks + wave * 32 * D), nlds = lds_address(nst), qlds = lds_address(Qs) + wave * 1024;
    const uint32_t kplace = klds + (c * D + ((h ^ swz<D>(c)) << 3)) * 2;      // operand ks of row c: 16-byte chunk 2 ks + h, at kplace ^ (ks << 5)

    // ---- the wave's list of blocks: of strip after strip, those beyond the last kHeldBlocks first, then these, then the first
    // ones again
    struct Cursor { int k, i, n, q0, again; };
    const int first_round = slot < a.missing ? 1 : 0;
    auto open = [&](Cursor& x) __attribute__((always_inline)) {      // the strip of round x.k: long and short ones in turn
        const int idx = x.k * a.n_slots + ((x.k & 1) ? a.n_slots - 1 - slot : slot) - a.missing;
        if (idx >= a.n_strips) { x.q0 = -1; x.n = 0; return; }
        x.q0 = 32 * idx;
        const int blocks = (min(a.S, x.q0 + 32) + 31) >> 5;
        x.n = max(0, (blocks - wave + NW - 1) / NW);
    };
    auto advance = [&](Cursor& x) __attribute__((always_inline)) {
        if (x.q0 < 0) return;
        ++x.i;
        const int early = x.n - kHeldBlocks;
        if (x.i < (x.again ? early : x.n)) return;
        x.i = 0;
        if (!x.again && early > 0) { x.again = 1; return; }
        x.again = 0;
        do { ++x.k; open(x); } while (x.q0 >= 0 && x.n == 0);
    };
    // (past the end of the list the first block is asked for: its stage has no reader)
    const int kkey = (int)(a.ks * 2), kstep = RPI * kkey, nkey = (int)(a.ns * nsz);       // bytes from key to key, request to request, row to row
    auto key_of = [&](const Cursor& x) __attribute__((always_inline)) { return x.q0 < 0 ? 0 : 32 * (wave + NW * x.i); };
    auto fetch_k = [&](uint32_t& at, int& so) __attribute__((always_inline)) {       // four requests, of NK
        request4<16, false, 1024>(krs, at, kvo[0], kvo[1], kvo[D == 128 ? 2 : 0], kvo[D == 128 ? 3 : 1], so, kstep);
    };
    auto noise_at = [&](const Cursor& x) __attribute__((always_inline)) { return max(x.q0, 0) * nkey + key_of(x) * nsz; };
    auto fetch_noise = [&](uint32_t& at, int& so) __attribute__((always_inline)) {   // four requests, of NN
        if constexpr (NB == 16) request4<16, NT, 1024>(nrs, at, nvo, nvo, nvo, nvo, so, 8 * nkey);
        else {
            request4<NB, false, 256>(nrs, at, nvo, nvo, nvo, nvo, so, nkey);
            so += 4 * nkey;                      // (rows 4 to 7 of eight are those of the other half of the lanes)
        }
    };
    const int qrow = (int)(a.qs * 2);
    auto fetch_q = [&](int q0) __attribute__((always_inline)) {      // eight requests or, of head_dim 64, four hold a strip's queries
#pragma unroll
        for (int i = 0; i < (D == 128 ? NQW : 1); ++i) {
            const int ln = lane_now(), row = (NW * i + wave) * RPI + ln / CPR;
            if (D == 128 || wave < 4) request1(qrs, qlds + i * NW * 1024, row * qrow + (((ln % CPR) ^ swz<D>(row)) << 4), q0 * qrow);
        }
    };

    // the noise runs two blocks ahead, K one: k_next is the key of the block that the noise was last asked for
    Cursor cn{first_round, 0, 0, 0, 0}, now{first_round, 0, 0, 0, 0};
    open(cn);
    if (cn.q0 >= 0 && cn.n == 0) { cn.i = -1; advance(cn); }
    open(now);
    fetch_q(max(now.q0, 0));
    auto fetch_block = [&](int stage) __attribute__((always_inline)) {
        uint32_t at = nlds + stage * 4096;
        int so = noise_at(cn);
#pragma unroll
        for (int i = 0; i < NN; i += 4) fetch_noise(at, so);
    };
    fetch_block(0);
    {
        uint32_t at = klds;
        int so = key_of(cn) * kkey;
#pragma unroll
        for (int i = 0; i < NK; i += 4) fetch_k(at, so);
    }
    advance(cn);
    fetch_block(1);
    int k_next = key_of(cn);
    advance(cn);
    int stage = 0;
    for (int i = tid; i < a.S + 31 && i < kKeys; i += NW * 64) Cs[i] = 0.f;
    wait_requests<2 * NN + NK>();
    wait_lds();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");

    constexpr float kNone = -3e38f;              // the reference of a row that has seen no finite score
    half8_t qA[NKS];
    float mlane = kNone, lsum = 0.f;             // of the one row a lane keeps: reference and sum
    auto row_of = [](int ln) __attribute__((always_inline)) { return 8 * ((ln & 15) >> 2) + 4 * (ln >> 5) + (ln & 3); };
    auto spread = [&](float x, float (&v)[16]) __attribute__((always_inline)) {      // the row's value from one lane to all
        const int ln = lane_now();
        float* const wr = Wr + wave * 32;
        wr[row_of(ln)] = x;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float4_t t = *reinterpret_cast<const float4_t*>(wr + 8 * i + 4 * (ln >> 5));
#pragma unroll
            for (int e = 0; e < 4; ++e) v[4 * i + e] = t[e];
        }
    };
    bool unseen = true;                          // some row's reference is still to come, or lies far below zero
    float16_t held[kHeldBlocks];

    // z - ref of a block, the rows' references being in wr; requests the blocks ahead.  All that can be done before the scores
    // are there is done between the MFMAs, which wait for each other.
    auto differences = [&](bool first, int q_next, int key0, int q0, float (&e)[16]) __attribute__((always_inline)) {
        wait_requests<NN>();                     // this block's K and noise: only the noise of the next was asked for behind them
        uint32_t at = kplace;
        if (D == 128) asm volatile("" : "+v"(at));      // (the eight places are not kept in registers)
        const float16_t zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        constexpr int NQ = 4;                    // operands in registers at a time
        half8_t kB[NQ];
#pragma unroll
        for (int ks = 0; ks < NQ; ++ks) kB[ks] = operand(at ^ (ks << 5));
        const float* np = nst + stage * 1024 + lane;
        const float* const rp = Wr + wave * 32 + 4 * h;
        float gn[16];
        float16_t s;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            if constexpr (NB == 2) gn[r] = (float)*reinterpret_cast<const half_t*>(np + 64 * r);
            else gn[r] = np[64 * r];
        }
        __builtin_amdgcn_sched_barrier(0);
        uint32_t kat = klds, nat = nlds + stage * 4096;
        int kso = k_next * kkey, nso = noise_at(cn);
        constexpr int READ = D == 128 ? NKS - NQ : 1;      // slot from which the stages have been read
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) {
            s = mfma32(qA[ks], kB[ks % NQ], ks == 0 ? zero : s);
            if (ks + NQ < NKS) kB[ks % NQ] = operand(at ^ ((ks + NQ) << 5));
            if (ks == READ) wait_lds();
            if (ks == READ && first) fetch_q(q_next);
            if (ks >= READ && ks < READ + NK / 4) fetch_k(kat, kso);
            if (ks == READ + NK / 4) {
#pragma unroll
                for (int i = 0; i < NN; i += 4) fetch_noise(nat, nso);
            }
            if (ks == READ + NK / 4) { k_next = key_of(cn); advance(cn); stage ^= 1; }
            if (ks >= NKS / 2) {
                constexpr int PER = 16 / (NKS / 2);
                const int first_r = (ks - NKS / 2) * PER;
#pragma unroll
                for (int r4 = first_r / 4; r4 < (first_r + PER) / 4; ++r4) {
                    const float4_t t = *reinterpret_cast<const float4_t*>(rp + 8 * r4);
#pragma unroll
                    for (int i = 0; i < 4; ++i) gn[4 * r4 + i] = __builtin_fmaf(gn[4 * r4 + i], a.c3, -t[i]);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) e[r] = __builtin_fmaf(s[r], a.c2, gn[r]);
        if (key0 + 31 > q0) {
            // the first of the strip's rows that sees the lane's key, counted from the lane's first row
            const int from = key0 + c >= a.S ? 64 : key0 + c - q0 - 4 * h;
#pragma unroll
            for (int r = 0; r < 16; ++r) e[r] = 8 * (r / 4) + (r % 4) >= from ? e[r] : -INFINITY;
        }
    };
    // The exponentials of a block relative to references (the first block's maxima) that only rise where a score exceeds them
    // by 64 -- in fp32 that costs no precision --; what was summed and held is scaled then.  With the reference zero, where the first block
    // allows it, a strip starts without the 32 lanes' maxima and two trips through LDS: whole calls, us, 71 heads of 64: 400 keys, fp32
    // 23.9 / 23.1, 777 fp16 44.3 / 42.2, 1536 fp32 111.7 / 111.4; 2 x 16, 1000 fp16 35.5 / 34.5.
    auto exponentials = [&](bool first, int q_next, int key0, int q0, int n_held, float (&e)[16], float* l) __attribute__((always_inline)) {
        differences(first, q_next, key0, q0, e);
        float top = max3(max3(e[0], e[1], e[2]), e[3], e[4]);
#pragma unroll
        for (int r = 5; r < 15; r += 2) top = max3(top, e[r], e[r + 1]);
        top = fmaxf(top, e[15]);
        if (D == 64 && first) {      // (no reference yet, and none is needed where all of the block lies within 64 of zero; head_dim 128 lacks the register)
            float far = max3(max3(fabsf(e[0]), fabsf(e[1]), fabsf(e[2])), fabsf(e[3]), fabsf(e[4]));
#pragma unroll
            for (int r = 5; r < 15; r += 2) far = max3(far, fabsf(e[r]), fabsf(e[r + 1]));
            if (__builtin_amdgcn_ballot_w64(!(fmaxf(far, fabsf(e[15])) <= 64.0f)) == 0) { mlane = 0.f; unseen = false; }
        }
        if (unseen || __builtin_amdgcn_ballot_w64(top > 64.0f) != 0) {
            float f[16];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float4_t t = *reinterpret_cast<const float4_t*>(Wr + wave * 32 + 8 * i + 4 * h);
#pragma unroll
                for (int j = 0; j < 4; ++j) e[4 * i + j] += t[j];
            }
            const float zmax = reduce_keys(e, lane_now(), [](float x, float y) __attribute__((always_inline)) { return fmaxf(x, y); });
            const float mn = mlane == kNone ? fmaxf(zmax, kNone) : zmax > mlane + 64.0f ? zmax : mlane;
            const float fl = fast_exp2(mlane - mn);
            spread(fl, f);
            lsum *= fl;
#pragma unroll
            for (int r = 0; r < 16; ++r)
                if (l) l[r] *= f[r];
#pragma unroll
            for (int i = 0; i < kHeldBlocks; ++i)
                if (i < n_held)
#pragma unroll
                    for (int r = 0; r < 16; ++r) held[i][r] *= f[r];
            mlane = mn;
            spread(mn == kNone ? 0.f : mn, f);
#pragma unroll
            for (int r = 0; r < 16; ++r) e[r] -= f[r];
            // A row whose reference lies far below zero -- its first keys masked by -1e4 or -1e9, say -- takes its next differences
            // from zero again: relative to that reference an ordinary score would be rounded to the reference's last place, and lost.
            const bool low = mn < -64.0f;
            unseen = __builtin_amdgcn_ballot_w64(low) != 0;
            if (low) Wr[wave * 32 + row_of(lane_now())] = 0.f;
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) e[r] = fast_exp2(e[r]);
    };

    for (; now.q0 >= 0; ++now.k, open(now)) {
        const int q0 = now.q0, n = now.n, early = max(0, n - kHeldBlocks), nh = n - early;
        Cursor nx{now.k + 1, 0, 0, 0, 0};
        open(nx);
        const int q_next = max(nx.q0, 0);
        uint32_t qat = kplace;
        asm volatile("" : "+v"(qat));            // (as above)
        qat += lds_address(Qs) - klds;
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) qA[ks] = operand(qat ^ (ks << 5));
        wait_lds();
        __builtin_amdgcn_s_barrier();            // every wave has its queries: the next strip's may come in
        asm volatile("" ::: "memory");
        if (n == 0) fetch_q(q_next);
        if (lane < 32) Wr[wave * 32 + lane] = 0.f;
        mlane = kNone; lsum = 0.f; unseen = true;
        const auto plus = [](float x, float y) __attribute__((always_inline)) { return x + y; };
        if (early > 0) {
            float l[16];
#pragma unroll
            for (int r = 0; r < 16; ++r) l[r] = 0.f;
            for (int i = 0; i < early; ++i) {
                float e[16];
                exponentials(i == 0, q_next, 32 * (wave + NW * i), q0, 0, e, l);
#pragma unroll
                for (int r = 0; r < 16; ++r) l[r] += e[r];
            }
            lsum = reduce_keys(l, lane_now(), plus);
        }
#pragma unroll
        for (int i = 0; i < kHeldBlocks; ++i)
            if (i < nh) {
                float e[16];
                exponentials(i == 0 && early == 0, q_next, 32 * (wave + NW * (early + i)), q0, i, e, nullptr);
#pragma unroll
                for (int r = 0; r < 16; ++r) held[i][r] = e[r];
            }
        // ---- the rows' normalisers, of all eight waves
        {
            float l[16];
#pragma unroll
            for (int r = 0; r < 16; ++r) l[r] = 0.f;
#pragma unroll
            for (int i = 0; i < kHeldBlocks; ++i)
                if (i < nh)
#pragma unroll
                    for (int r = 0; r < 16; ++r) l[r] += held[i][r];
            lsum += reduce_keys(l, lane_now(), plus);
        }
        const int row = row_of(lane_now());
        St[wave * 32 + row] = float2_t{mlane, lsum};
        if (n == 0) wait_requests<0>(); else wait_requests<NK + NN>();      // the next strip's queries
        wait_lds();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        float mx = kNone, ls = 0.f;
#pragma unroll
        for (int half = 0; half < NW; half += 4) {
            float2_t st[4];
            float top = mx;
#pragma unroll
            for (int w = 0; w < 4; ++w) { st[w] = St[(half + w) * 32 + row]; top = fmaxf(top, st[w][0]); }
            ls *= fast_exp2(mx - top);
            mx = top;
#pragma unroll
            for (int w = 0; w < 4; ++w) ls = __builtin_fmaf(st[w][1], fast_exp2(st[w][0] - mx), ls);
            __builtin_amdgcn_sched_barrier(0);
        }
        const float lse2 = mx + fast_log2(ls);
        const bool real = q0 + row < a.S;
        if (wave == 0 && (lane & 16) == 0 && real) a.lse[((int64_t)b * a.Hq + head) * a.S + q0 + row] = lse2 * kLn2;
        // ---- the held blocks' column sums.  (Weights without lse2, whose rounding at 1e8 and more would be a factor.  A row without
        // a normaliser -- no finite score, or +inf or NaN among them -- makes a NaN of every key that it sees; of the others, whose
        // exponentials are zeros, it must not: they are left out where a block has any.)
        float w[16];
        spread(real ? fast_exp2(mlane - mx) * __builtin_amdgcn_rcpf(ls) : 0.f, w);
#pragma unroll
        for (int i = 0; i < kHeldBlocks; ++i)
            if (i < nh) {
                const int key0 = 32 * (wave + NW * (early + i));
                float x = held[i][0] * w[0];
                if (key0 == q0) {
                    const int ln = lane_now(), from = (ln & 31) - 4 * (ln >> 5);      // (compared here and not once for all blocks)
                    if (from > 0) x = 0.f;
#pragma unroll
                    for (int r = 1; r < 16; ++r) x = 8 * (r / 4) + (r % 4) >= from ? __builtin_fmaf(held[i][r], w[r], x) : x;
                } else {
#pragma unroll
                    for (int r = 1; r < 16; ++r) x = __builtin_fmaf(held[i][r], w[r], x);
                }
                x = half_sum(x);
                if (h == 0) Cs[key0 + c] += x;
            }
        // ---- ... and the others', once more from K and the noise
        if (early > 0) {
            Wr[wave * 32 + row] = real ? lse2 : INFINITY;
            for (int i = 0; i < early; ++i) {
                const int key0 = 32 * (wave + NW * i);
                float e[16];
                differences(false, 0, key0, q0, e);
                float x = 0.f;
#pragma unroll
                for (int r = 0; r < 16; ++r) x += fast_exp2(e[r]);
                x = half_sum(x);
                if (h == 0) Cs[key0 + c] += x;
            }
        }
    }
    wait_requests<0>();                          // (nothing lands in these stages once they are given up)
    const int64_t bh = (int64_t)b * a.Hq + head;
    if (lane < 32)
        for (int key = 32 * wave + c; key < a.S; key += 32 * NW) {
            if (a.n_slots == 1) store_stat(a.out, a.s16, bh * a.S + key, Cs[key]);
            else a.part[(bh * a.n_slots + slot) * a.S + key] = Cs[key];
        }
#endif
}

__global__ __launch_bounds__(256) void attn_add_slots_kernel(const SlotSums a) { add_slots(a, (int64_t)blockIdx.x * 256 + threadIdx.x); }
hipError_t launch_add_slots(const SlotSums& a, hipStream_t s) {
    hipLaunchKernelGGL(attn_add_slots_kernel, dim3((unsigned)((a.n + 255) / 256)), dim3(256), 0, s, a);
    return hipGetLastError();
}

// Two workgroups of four waves a CU instead of one of eight: the waves that wait for the end of a strip are then half as many,
// and the other workgroup's go on; but 1024 held keys instead of 2048.  us, four / eight waves: 71 heads of 64: 600 33.4 / 41.0,
// 1536 113 / 124, 2050 243 / 235; 32 of 128: 1024 48.7 / 50.3, 1501 91.6 / 89.1; 16 of 64: 1100 43.9 / 37.3, 1536 50.3 / 44.2.
static int strip_waves(const trn_attn_desc* d) {
    return (int64_t)d->batch * d->n_q_heads >= 32 && d->seq_q + 31 <= strip_keys(4, 128) ? 4 : 8;
}

// Workgroups per head: a workgroup's time is its start and its share of the head's strips, and the chip takes so many at once.  fill: of these places
// in all rounds, the percentage that is taken.
static int strip_slots(const trn_attn_desc* d, int64_t& fill) {
    const int waves = strip_waves(d);
    const int64_t bh = (int64_t)d->batch * d->n_q_heads, at_once = waves == 8 ? 256 : 512;
    const int n_strips = (d->seq_q + 31) / 32;
    const double work = 0.06 * n_strips * (n_strips + 1) + 0.7 * n_strips, start = 3.0;      // (us)
    int best = 1;
    double least = 1e30;
    for (int n = 1; n <= n_strips && n <= 64; ++n) {
        const double t = (double)((bh * n + at_once - 1) / at_once) * (start + work / n) + 0.02 * n;
        if (t < least) { least = t; best = n; }
    }
    fill = bh * best * 100 / ((bh * best + at_once - 1) / at_once * at_once);
    return best;
}

// Where this launch and the plain attention, which adds the sums of a head's workgroups, are faster than the forward with noise and the
// column statistics: causal prompts nearly throughout, but not
//   -- the longest rows, of which 2048 keys are held and the rest is read and multiplied twice;
//   -- fp16 noise, half as much to read for the same arithmetic, of long rows of few heads;
//   -- long prompts of 64 to 319 heads with keys of their own, when the heads' count is no multiple of the 8 XCDs: a head's
//      workgroups are then on all of them, and each L2 reads all of K.  With head_dim 128, whose K is the larger, so are from some length
//      on those of more than 16 KV heads in all that are no multiple;
//   -- short prompts of 171 to 255 heads: the chip takes two workgroups a head at once, but not three, and two leave up to a third of it
//      idle.  With head_dim 128 and fp16 noise, where there is the least to gain, so it is with every number of 128 heads and more that leaves
//      a fifth of the places empty (an eighth, from 256 on), and with 48 KV heads in all that are no multiple, or 64.
// Calls one after the other, here / two passes in per cent of time (2500 sizes; minus: faster here):
//   D = 64, fp32   71 heads: 420 keys -8, 1001 -30, 2600 -20; 128: 200 -8, 289 -5; 160: 208 -2, 240 +1, 272 -15; 284: 200 -3, 272 -21; 320: 240 -18; 16: 1000 -39, 2100
//         -18.  Left out: 176, 202 +18, 256 +9; 192, 208 +14; 224, 202 +14; 256, 200 to 225 (kept) +6 to +1, 256 -9; 4800 keys: 12 heads +10, 16 -3, 8 (kept) -7
//   D = 64, fp16   71: 520 -19, 1000 -17, 2600 -8; 20: 1440 -25; 32: 1500 -4, 2000 -7, 3000 -9; 48: 1360 -11, 1700 -1, 2400 -11; 142: 380 -6, 560 -14; 192: 385 -4, 530 -4, 650
//         -14.  Left out: 176 to 192, 420 to 500 +3 to +9; 284, 330 +1, 568, 290 +6; 24 heads, 1700 to 2000 +1 to +8 (1500 -11); 16, 2600 +9, 3300 +13; 142 with keys of
//         their own, 1650 +9
//   D = 128, fp32  32: 420 -17, 1000 -21, 2100 -13, 3210 -7, 3790 -2; 64: 160 -40, 260 -7, 2400 -8, 3790 -4; 256: 260 -14, 1400 -19; 24: 420 -23, 1300 -7, 3600 -6; 18: 3401
//         -10, 3900 -17; 20: 3401 -19, 4000 (kept) +3; 28: 3450 -9; 100 on 25 KV heads: 1350 -4; 16: 520 -13, 1300 -29; 10: 520 -22; 8: 1800 -29, 4000 -17.  Left out: 256, 200
//         +5; 37 with keys of their own, 3777 +27, 39, 3186 +12, 40, 3648 +11, 56, 2944 +8, 34 on 17, 3619 +9; 26, 3800 to 4150 +5, 30, 3401 to 4150 +2 to +11; 32, 4000 +5; 16 heads, 2700 to 3640 +3 to +9; 100 on 25, 2000 +6, 136 on 34 +3; 142 with keys of their own,
//         1190 to 1500 +1 to +15
//   D = 128, fp16  32: 420 -15, 1000 -15; 8: 1000 -16, 2600 -30, 4000 -18; 16: 520 -11, 1000 -27; 9: 900 -3; 48: 360 -6, 1400 -7; 80: 430 -8, 1300 -1; 112: 430 +3, 830 -11,
//         1300 -6; 128: 530 -13, 1590 -4; 192: 700 -3, 1300 -8; 256: 640 -11, 1300 -13, 2500 -5; 155: 411 -14; 204: 650 -9; 336: 534 -8; 300: 780 -9; 480: 918 -11; 168 with keys of their own: 538 -10; 100 on 25: 1050 -8; 71 with keys of their own: 520 -7, 800 +3, 100: 800 -11.  Left out:
//         32, 1350 +4, 1800 +5; 48, 1700 +6; 96, 1500 +3; 80, 1700 +10; 128, 1700 +4, 2500 +3; 160, 1700 +7; 176, 450 +14, 545 +5; 192, 500 +11; 88 on 22, 1391 +5; 100 on 25, 1350 +7; 200 on 50 +8; 71 with
//         keys of their own, 1200 +8; 77, 838 +6, 95, 745 +9; 142, 520 +3, 1200 +17; 189 on 63, 941 +16; 264 on 24, 496 +13, 288, 554 +8, 312, 1223 +8, 405, 638 +8; 264 to 495 of their own +1 to +17; 16, 2200 +2, 2700 to 3640 +6 to +17; 8 and 9, 4400 +5
// Short prompts of these lines, where a launch counts: 70 of 128, 210, fp16 -37; 40 of 64, 226, fp32 -28; 48 of 64, 240, fp16 -29; 40 of 128, 180, fp16 -5.
// (Not for speed: prompts of 65 to 127 heads of 64 below 300 keys and of up to 16 heads with less noise than these lines ask for would gain 2 to 17 %
// too.  That 71 heads of 64 with 299 keys, 16 with 600 and 8 of 128 with 600 have no workspace is what a test of these lines has held fast from the first.)
static bool strips_suit(const trn_attn_desc* d, bool n16) {
    if (!d->causal || d->seq_q != d->seq_kv || d->seq_q < 160) return false;
    const int64_t bh = (int64_t)d->batch * d->n_q_heads, bkv = (int64_t)d->batch * d->n_kv_heads, mb = (bh * d->seq_q * d->seq_q * (n16 ? 1 : 2)) >> 20;
    const int64_t strips = bh * ((d->seq_q + 31) / 32), S = d->seq_q;
    const bool second_strips = bh <= 16 && strips > 256 && strips <= 320;
    const bool scattered = bh % 8 != 0 && bh < 320 && bkv >= 64, uneven = bkv % 8 != 0 && bkv > 16;
    if (d->head_dim == 64) {
        if ((second_strips && S <= 1024) || (S > 4500 && bh > 8)) return false;
        const bool launches = S >= 200 && bh >= 18 && bh <= 64;
        if (!n16) return launches || (S < 300 ? S >= (bh > 170 && bh < 256 ? 257 : 200) && bh >= 128 : mb >= 12);
        if (S > 1250 && !(bh < 22 ? mb <= 96 : bh >= 32 && !scattered)) return false;
        return launches || (S >= 300 && mb >= 7 && (bh <= 80 || S >= 380) && !(bh > 170 && bh < 205 && S > 416 && S <= 512));
    }
    if (S > 4200) return false;
    if (n16) {
        if (bh <= 16) return S >= 300 && mb >= 4 && (bh <= 8 || mb <= (bh <= 10 ? 95 : 70));
        if (S < (bh <= 64 ? 180 : bh <= 128 ? 240 : bh > 170 && bh < 205 ? 561 : 420)) return false;
        if (bh < 40) return mb <= 44;
        if (bh < 128) return S <= (scattered ? (bh < 76 ? 900 : bh < 88 ? 780 : 560) : uneven ? 1200 : 1400);
        if (bkv >= 64) return bh % 8 == 0 && bkv % 8 == 0 && bh < 176 && S <= 1000;
        if (bkv >= 48 && bkv % 8 != 0) return false;
        int64_t fill;
        strip_slots(d, fill);
        if (bh < 256) return fill >= 80 && S <= (fill >= 99 ? 1600 : bkv < 32 ? 1300 : 900);
        return fill >= 87 && S <= (fill >= 99 ? 2600 : 1000);
    }
    if (scattered && S > 700) return false;
    if (S < 300) return bh >= 18 && S >= (bh < 64 ? 180 : bh < 192 ? 160 : 260);
    if (bh >= 18) return mb <= 640 || (!uneven && S <= (bh < 32 ? 3400 : bh > 32 && bkv == bh ? 2500 : 3800));
    return mb >= (bh > 8 ? 3 : 16) && (bh <= 12 || mb <= 200);
}
int noise_strip_slots(const trn_attn_desc* d, bool n16) {
    int64_t fill;
    return strips_suit(d, n16) && d->seq_q + 31 <= strip_keys(strip_waves(d), d->head_dim) ? strip_slots(d, fill) : 0;
}

// A head's strips are dealt to its workgroups in rounds of n_slots, in turns of direction.  Where the last round is not full, strips
// are taken as missing from the first one, the shortest, instead of from the last, the longest: the sums of strips are then equal
// after an even number of rounds, and a short strip apart after an odd one.  Of two workgroups a CU, whose sum counts, the odd numbers
// gain little, and of more than 56 heads nothing.  us, missing from the last / first: one workgroup: 8 of 64: 2170 keys 49.0 / 41.3; 8 of 128: 2103
// 60.6 / 51.1; 16 of 64: 2116 75.2 / 65.4; 32 of 64: 1600 69.6 / 56.3; 40 of 64: 2327 179 / 163; 64 of 64: 3337 512 / 491; 71 of 64: 2600 342 / 332; two, even: 32 of 128: 514
// 30.8 / 24.7, 1600 95.4 / 83.3; 64 of 128: 1300 107 / 97; 48 of 128: 993 -11 %; 71 of 64: 777 39.7 / 37.9; odd: 44 of 128: 1603 130 / 123; 40 of 64: 953 35.9 / 37.6; left out:
// 64 of 64: 578 28.9 / 30.2; 80: 1227 +8 %; 71: 948 53.1 / 54.5, 601 31.6 / 30.8.
static int strips_missing(const trn_attn_desc* d, int n_strips, int n_slots) {
    const int rounds = (n_strips + n_slots - 1) / n_slots;
    if (strip_waves(d) == 4 && (int64_t)d->batch * d->n_q_heads > 56 && (rounds & 1)) return 0;
    return rounds * n_slots - n_strips;
}

int64_t noise_strips_workspace_bytes(const trn_attn_desc* d, int with_noise) {
    const int n32 = with_noise == 2 ? 0 : noise_strip_slots(d, false), n16 = with_noise == 3 ? 0 : noise_strip_slots(d, true);
    const int64_t n = n32 > 0 ? n32 : n16;       // (the same number where both suit)
    return n <= 1 ? 0 : n * d->batch * d->n_q_heads * d->seq_kv * 4;         // (one workgroup a head writes its sums itself)
}

template <int D, int NW>
static void launch_strips(const StripArgs& a, int nb, bool nt, unsigned grid, hipStream_t s) {
    const dim3 g(grid), t(NW * 64);
    if (nb == 2) hipLaunchKernelGGL((attn_noise_strips_kernel<D, 2, false, NW>), g, t, 0, s, a);
    else if (nb == 4) hipLaunchKernelGGL((attn_noise_strips_kernel<D, 4, false, NW>), g, t, 0, s, a);
    else if (nt) hipLaunchKernelGGL((attn_noise_strips_kernel<D, 16, true, NW>), g, t, 0, s, a);
    else hipLaunchKernelGGL((attn_noise_strips_kernel<D, 16, false, NW>), g, t, 0, s, a);
}

hipError_t launch_noise_strips(const trn_attn_desc* d, const void* q, const void* k, const void* noise, bool n16, float* lse, void* out,
                               bool s16, void* workspace, SlotSums& left, hipStream_t s) {
    StripArgs a;
    a.q = (const half_t*)q; a.k = (const half_t*)k; a.noise = noise; a.lse = lse; a.out = (float*)out; a.part = (float*)workspace;
    a.B = d->batch; a.Hq = d->n_q_heads; a.Hkv = d->n_kv_heads; a.S = d->seq_q;
    a.heads = HeadMap(a.B, a.Hq, a.Hkv);
    a.n_strips = (d->seq_q + 31) / 32; a.n_slots = noise_strip_slots(d, n16); a.missing = strips_missing(d, a.n_strips, a.n_slots);
    a.qb = d->q_stride_b; a.qh = d->q_stride_h; a.qs = d->q_stride_s;
    a.kb = d->k_stride_b; a.kh = d->k_stride_h; a.ks = d->k_stride_s;
    a.nb = d->noise_stride_b; a.nh = d->noise_stride_h; a.ns = d->noise_stride_s;
    a.c2 = d->scale * kLog2e / d->tau; a.c3 = kLog2e / d->tau;
    a.s16 = s16 ? 1 : 0;
    const int64_t bh = (int64_t)a.B * a.Hq;
    const bool grid16 = aligned16(noise) && pitch16(a.ns, 4) && pitch16(a.nh, 4) && pitch16(a.nb, 4);
    const int nb = n16 ? 2 : grid16 ? 16 : 4;
    const bool nt = (reinterpret_cast<uintptr_t>(noise) & 127u) == 0 && !(a.ns & 31) && !(a.nh & 31) && !(a.nb & 31);
    const unsigned grid = (unsigned)(bh * a.n_slots);
    const bool wide = strip_waves(d) == 8;
    if (d->head_dim == 128) { if (wide) launch_strips<128, 8>(a, nb, nt, grid, s); else launch_strips<128, 4>(a, nb, nt, grid, s); }
    else { if (wide) launch_strips<64, 8>(a, nb, nt, grid, s); else launch_strips<64, 4>(a, nb, nt, grid, s); }
    left = SlotSums{a.part, out, bh * a.S, a.n_slots > 1 ? a.n_slots : 0, a.S, a.s16, Div(a.S)};
    return hipGetLastError();
}

}  // namespace trn
