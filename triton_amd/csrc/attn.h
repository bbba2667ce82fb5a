// Argument block shared by the attention forward kernels.
#pragma once
#include "common.h"

namespace trn {

// Column sums of a head's workgroups that are still to be added, in their order: part [heads][n_slots][keys] fp32 into out
// [heads][keys] (KeyFormer's single pass: attn_noise_strips.hip).  n_slots = 0: none.
struct SlotSums { const float* part; void* out; int64_t n; int n_slots, keys, s16; Div by_keys; };

struct AttnArgs {
    const half_t* q; const half_t* k; const half_t* v; half_t* o;
    float* lse; const half_t* gamma_q; const float* noise; float* lse_pert;
    int B, Hq, Hkv, Sq, Skv, n_qtiles;
    HeadMap heads;
    int pack;      // prefill kernels: 2^pack heads of a KV head to a workgroup (attn_fwd16.hip)
    int even;      // prefill kernels with split keys: two tiles of 64 queries a workgroup (attn_fwd16.hip)
    int64_t qb, qh, qs, kb, kh, ks, vb, vh, vs, ob, oh, os, nb, nh, ns;
    float c1;      // scale * log2(e)                    : plain scores in the log2 domain
    float c2, c3;  // scale*log2(e)/tau, log2(e)/tau     : perturbed scores  z2 = s*c2 + g*c3
    float q_eps;
    int causal, q_norm;
    const half_t* gamma_k; float k_eps; int k_norm;     // decode kernel without noise only: the keys are normalised on arrival
    // decode kernel only: keys split over n_split workgroups per head, partial results and arrival counters in ws
    int n_split;
    int partial;   // ... which the next launch merges (2: of the queries there are alone)
    int spread;    // decode kernel only: the query tiles of a head go to all XCDs
    float* ws;
    // decode kernel only, at most 32 queries: per-key sums (and sums of squares) of the probabilities -- of the
    // perturbed ones when noise is given -- from a second sweep over the keys once the row normalisers are final
    float* col_sum; float* col_sumsq;
    int mean_std;  // short kernel, and decode kernel with shared-out keys: ... turned into mean and standard deviation
    // ... and the probabilities themselves, un-reduced: float [B, Hq, Sq, Skv] contiguous
    float* probs;
    int n16;       // noise points at fp16 data (its pitches count halfs; any alignment: see HalfNoise)
    int s16;       // decode and short kernels: col_sum and col_sumsq point at fp16 data
    int o_nt;      // prefill kernels: the output goes past the caches (outputs_stream)
    SlotSums sums; int n_main;     // prefill kernels with the queries as given: sums to add, by the workgroups from n_main on
};

// Whether a launch of so many outputs stores them past the caches.  What it leaves dirty in the L2s is written back before it ends, on
// top of the launch; but the output projection behind an attention reads what the caches still hold.  us, through the caches / past them:
//   the launch alone: 32 heads of 128: 4 x 777 tokens (25 MB) 36.1 / 33.1, 8 x 500 34.3 / 30.4, 4096 122.2 / 117.7; 71 of 64, 2048 (19 MB) 46.0 / 45.6
//   projection of Q, K, V, attention, output projection by the library's product; by ours (runs of one side differ by 1 %):
//     small ones lose: 32 heads of 128, 300 tokens (2.5 MB) 82.3 / 82.3; 67.0 / 70.5, 777 (6 MB) 127.2 / 127.1; 120.7 / 122.8; 71 of 64, 400 (4 MB) 81.8 / 83.9;
//       72.0 / 83.8; 16 of 64, 1000 (2 MB) 37.2 / 39.6; 35.5 / 36.0
//     from 8 MB on they are the same: 1442 (12 MB) 173.8 / 173.7; 189.0 / 187.9, 2048 (17 MB) 219.7 / 221.9; 241.2 / 242.1; 71 of 64, 1000 (9 MB) 149.6 / 150.9;
//       172.9 / 171.8, 2048 262.0 / 261.2; 267.0 / 263.3, 4 x 777 396.4 / 394.2; 508.3 / 507.0; 16 of 64, 8 x 1000 (16 MB) 121.3 / 121.2; 130.8 / 129.6; with
//       KeyFormer's scores, fp32 noise, 2048 311.9 / 311.8; 330.5 / 329.9, 71 of 64, 1442 289.0 / 287.5; 295.9 / 295.9
inline bool outputs_stream(int64_t rows, int head_dim) { return rows * head_dim * 2 >= (int64_t)8 << 20; }
template <class V> __device__ __forceinline__ void store_out(void* p, V v, int past) {
    if (past) {
        asm volatile("" ::: "memory");      // (the two stores would be merged into one without the hint)
        __builtin_nontemporal_store(v, static_cast<V*>(p));
        asm volatile("" ::: "memory");
    } else *static_cast<V*>(p) = v;
}

// fp16 noise as the kernels fetch it.  Its rows may start at any element (the reference's [.., M, P + M] tensors have any
// key count), so a lane reads the whole dwords around its 4 keys -- three of them cover both cases -- and shifts by half a
// dword where its row starts on an odd element.  Nothing outside the dword that holds a row's last key is ever read: the
// base is rounded down to a dword and the range up to one.
#if defined(__HIP_DEVICE_COMPILE__)
typedef uint32_t uint3_t __attribute__((ext_vector_type(3)));
struct HalfNoise {
    __amdgpu_buffer_rsrc_t rs;
    int odd;           // 1: the base was rounded down by one element
    __device__ __forceinline__ HalfNoise(const void* head_base, int64_t rows, int64_t pitch, int64_t cols) {
        const uintptr_t p = reinterpret_cast<uintptr_t>(head_base);
        odd = (int)(p >> 1) & 1;
        rs = __builtin_amdgcn_make_buffer_rsrc((void*)(p & ~(uintptr_t)3), 0, (int)((((rows - 1) * pitch + cols + odd) * 2 + 3) & ~3), 0x00020000);
    }
    // byte offset of a row's (rounded down) start and the shift of its elements within the dwords
    __device__ __forceinline__ int row(int64_t first_elem, int& shift) const {
        const int64_t e = first_elem + odd;
        shift = (int)(e & 1) * 16;
        return (int)((e & ~(int64_t)1) * 2);
    }
};
// the 4 values out of three dwords
__device__ __forceinline__ half4_t half_noise4(const uint3_t& d, int shift) {
    const uint2_t u = {__builtin_amdgcn_alignbit(d.y, d.x, shift), __builtin_amdgcn_alignbit(d.z, d.y, shift)};
    return __builtin_bit_cast(half4_t, u);
}
#endif

// A wave's per-key sums, 16 per lane over the lane's queries, added up over the 32 lanes of each half through 4 KB of LDS:
// lane 2k + i gets key number k of the wave's 32 from 16 lanes (each key starting at another one: no bank conflicts) and
// adds its neighbour's.  (In registers, five exchanges of all 16 sums and a division per sum and lane behind them took
// 1 - 2 us of a launch.)
// (lo, hi: the first and the second 2 KB)
__device__ __forceinline__ void put_sums(const float (&v)[16], float* lo, float* hi, int lane) {
#pragma unroll
    for (int r = 0; r < 8; ++r) { lo[r * 64 + lane] = v[r]; hi[r * 64 + lane] = v[8 + r]; }
}
__device__ __forceinline__ float key_sum(const float* lo, const float* hi, int lane) {
    const float* area = lane < 32 ? lo : hi - 512;
    const int kh = (lane >> 1) & 1, r = lane >> 2, part = lane & 1;        // the key's half kh and number r of 16
    float x[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) x[i] = area[r * 64 + kh * 32 + part * 16 + ((i + r) & 15)];
#pragma unroll
    for (int n = 8; n >= 1; n >>= 1)                                       // (as a tree: a chain's rounding is larger)
#pragma unroll
        for (int i = 0; i < n; ++i) x[i] += x[i + n];
    return x[0] + __shfl_xor(x[0], 1, 64);
}
// The key, of the block's 32, that a lane has from key_sum.
__device__ __forceinline__ int key_of_sum(int lane) {
    const int kh = (lane >> 1) & 1, r = lane >> 2;
    return 8 * (r / 4) + 4 * kh + (r % 4);
}
// The sums x, y of a key's probabilities and their squares over the n queries that see it, into mean and standard deviation.
__device__ __forceinline__ void mean_std_of(float& x, float& y, float n) {
    const float mean = x / n;
    // E p^2 - mean^2 as (y - x mean) / n, the product fused.  The difference is known to about 1e-7 of E p^2, its
    // root to 3e-4 of the column's root mean square: a key seen by a single query, whose spread is zero by
    // definition, would come back as that rounding residue, so it is set.
    y = n > 1.5f ? __builtin_sqrtf(fmaxf(0.f, __builtin_fmaf(-x, mean, y) / n)) : 0.f;
    x = mean;
}
// (fp16: the fp32 value rounded once, as a copy into the caller's tensor would)
__device__ __forceinline__ void store_stat(float* out, int s16, int64_t at, float v) {
    if (!out) return;
    if (s16) reinterpret_cast<half_t*>(out)[at] = (half_t)v;
    else out[at] = v;
}

// One element a thread.
__device__ __forceinline__ void add_slots(const SlotSums& a, int64_t i) {
    if (i >= a.n) return;
    const int bh = a.by_keys.of((int)i), key = (int)i - bh * a.keys;
    const float* p = a.part + (int64_t)bh * a.n_slots * a.keys + key;
    float x = 0.f;
    for (int s = 0; s < a.n_slots; s += 8) {     // (eight on their way at once.  Whole calls, us, one after the other / so: 8 heads of 128, 4096 keys (32
                                                 // slots) 144.3 / 137.8; 16 of 64, 1536 41.9 / 39.4; 32 of 128, 1024 44.6 / 41.9)
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = p[(int64_t)min(s + e, a.n_slots - 1) * a.keys];
#pragma unroll
        for (int e = 0; e < 8; ++e) x += s + e < a.n_slots ? v[e] : 0.f;
    }
    store_stat(static_cast<float*>(a.out), a.s16, i, x);
}

// Checks, argument block and kernel choice behind every attention entry point of the C ABI.  given_q: without noise too the queries
// are not multiplied by the scale, and rounded, before the products (attn_fwd16.hip; the other kernels never do).  sums: taken along by the
// same launch, or added by one behind it.  check_only: nothing is launched.
int attn_forward(const trn_attn_desc* d, const void* q, const void* k, const void* v, void* o, float* lse,
                 const void* gamma_q, const float* noise, float* lse_pert, void* workspace,
                 int64_t workspace_bytes, float* col_sum, float* col_sumsq, void* stream, float* probs = nullptr,
                 bool n16 = false, bool s16 = false, bool any_pitch = false, bool k_norm = false, const void* gamma_k = nullptr,
                 float k_eps = 0.f, bool mean_std = false, bool given_q = false, const SlotSums* sums = nullptr, bool check_only = false);

// The checks of attn_colstats by themselves, for a caller that launches something else before it.
int attn_colstats_check(const trn_attn_desc* d, const void* q, const void* k, const float* lse, const float* noise,
                        const float* out_sum, const float* out_sumsq, bool n16, bool any_pitch);

// Checks, argument block and kernel choice behind the column statistics (attn_colstats.hip); mean_std: the two outputs
// are the mean and standard deviation; n16 / s16: fp16 noise / outputs; any_pitch: fp32 noise on any dword (16-byte
// buffer loads need no more).
int attn_colstats(const trn_attn_desc* d, const void* q, const void* k, const float* lse, const float* noise, float* out_sum,
                  float* out_sumsq, int mean_std, void* stream, bool n16 = false, bool s16 = false, bool any_pitch = false);

// Whether the kernels that read all of this noise request it past the caches (attn_fwd.hip).
bool noise_streams(const trn_attn_desc* d, const void* noise, bool n16);

// KeyFormer's row normalisers and key scores in one pass over the noise (attn_noise_strips.hip): in how many workgroups per head
// (0: this problem does not suit it), and with how much workspace, of any contents, for noise of either type (1), fp16 (2), fp32 (3); none with one workgroup a head.
int noise_strip_slots(const trn_attn_desc* d, bool n16);
int64_t noise_strips_workspace_bytes(const trn_attn_desc* d, int with_noise);
hipError_t launch_noise_strips(const trn_attn_desc* d, const void* q, const void* k, const void* noise, bool n16, float* lse, void* out,
                               bool s16, void* workspace, SlotSums& left, hipStream_t s);       // left: what the caller has to have added
hipError_t launch_add_slots(const SlotSums& a, hipStream_t s);

// One workgroup per head and 32 queries, whose eight waves split the keys (attn_decode.hip): at most 32 queries per head
// (decode), and problems with so few query tiles that the prefill kernels would leave most of the chip idle.
bool attn_decode_suits(int batch, int n_q_heads, int seq_q, int seq_kv, int head_dim, bool causal, bool noise);
hipError_t launch_attn_decode(AttnArgs a, int head_dim, void* workspace, int64_t workspace_bytes, hipStream_t stream);
// ... and where that launch, without a workspace, also normalises the keys if asked to (args.k_norm).
bool attn_decode_norms_keys(int batch, int n_q_heads, int seq_q, int seq_kv, int head_dim);
const char* attn_decode_kernel_name(int batch, int n_q_heads, int seq_q, int seq_kv, int head_dim, bool noise);
// Bytes of workspace with which launch_attn_decode splits the keys of this problem over several workgroups (0: it would not).
int64_t attn_decode_workspace_bytes(int batch, int n_q_heads, int seq_q, int seq_kv, int head_dim);
int64_t attn_few_query_workspace_bytes(int batch, int n_q_heads, int n_kv_heads, int seq_q, int seq_kv, int head_dim);      // ... where that is 0, for two launches

// ... and of that with which it does for key statistics, merged and summed up by a second launch.
int64_t attn_decode_stats_workspace_bytes(int batch, int n_q_heads, int seq_q, int seq_kv, int head_dim, bool noise);
// ... over how many workgroups a head with a workspace of so many bytes (0: the statistics are part of a single launch).
int attn_decode_stat_shares(int batch, int n_q_heads, int n_kv_heads, int seq_q, int seq_kv, int head_dim, bool noise, int64_t workspace_bytes);

// Device address, on the current device, of the library's static scratch array (TRN_ATTN_NOALLOC_SCRATCH_BYTES bytes)
// behind trn_attn_fwd_noalloc_f16; looked up once per device.  nullptr if the runtime refuses.
void* attn_static_scratch();

// Attention and key statistics of at most 128 queries and keys in one launch (attn_short.hip).
bool attn_short_suits(int seq_q, int seq_kv);
hipError_t launch_attn_short(const AttnArgs& a, int head_dim, hipStream_t s);

// The forward pass without score perturbation on the 16x16x32 MFMA (attn_fwd16.hip).  Narrow: 4 waves x 32 queries
// per workgroup; Wide: 8 waves x 32 consecutive queries; Paired: 8 waves, two 128-query tiles from opposite ends of
// the sequence (causal problems whose grid is a single round); Split: 8 waves on 128 queries, two groups of four that
// take every other 64-key tile each (small grids, long walks), of a causal problem 64 from either end.
enum class Attn16Shape { Narrow, Wide, Paired, Split };
Attn16Shape attn_fwd16_shape(int batch, int n_q_heads, int seq_q, int seq_kv, int head_dim, bool causal);
hipError_t launch_attn_fwd16(const AttnArgs& a, int head_dim, Attn16Shape shape, bool given_q, hipStream_t stream);
// The keys of a chunk of queries against a long cache shared out over workgroups (attn_fwd16.hip): fp32 partial results in
// args.ws, attn_share_workspace_bytes of it (0: this problem is not shared out), merged by a second launch.
int64_t attn_share_workspace_bytes(int batch, int n_q_heads, int seq_q, int seq_kv, int head_dim);
hipError_t launch_attn_shares(const AttnArgs& a, int head_dim, hipStream_t stream);
// Name of the kernel instantiation that launch_attn_fwd16 runs for this shape, as a profiler prints it.
const char* attn_fwd16_kernel_name(int head_dim, Attn16Shape shape);

}  // namespace trn
