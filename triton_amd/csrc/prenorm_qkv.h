// Argument block shared by the two tile shapes of the fused RMSNorm + Q/K/V projection GEMM.
#pragma once
#include "common.h"

namespace trn {

// One projection: weight [hidden][n] with row pitch ldw, head-split output, the index of its first column panel in
// the concatenated [Q | K | V] panel list, and an optional addend laid out like the output (out = x w + addend; it
// may be the output itself).  n = 0: no such projection.
struct ProjOut { const half_t* w; half_t* out; int64_t ldw, stride_h, stride_s; int n; int tile0; const half_t* addend; };

// Panels are GBN (128) or WN (256) columns wide depending on the kernel; n_mtiles counts token tiles likewise.
struct GemmArgs {
    const half_t* x; const half_t* gamma;
    ProjOut p[3];
    int T, K, head_dim, n_mtiles, n_panels, panels_per_xcd;
    int64_t ldx;
    float eps;
    int norm;
};

// Chunk swizzle of a W stage row (16-byte chunks) as a function of the row: a bit permutation of the row's low
// 4 bits, XORed into the low 4 bits of the chunk index, under which 4 consecutive rows read over 4 consecutive
// chunks (one phase of the transposing read) touch every bank once.
__device__ __forceinline__ int wswz(int r) { return ((r & 3) << 2) | ((r >> 2) & 3); }

// Whether weights that one workgroup each reads once are requested past the caches (the non-temporal hint): 64 MB and more,
// of which the last-level cache (256 MB) keeps nothing until the same layer comes round again but would evict what it holds
// for each line.  us, without / with, weights and cache cold (three sets in turn): whole decode step, 16 tokens on 1024, 4096 ->
// 12288 (101 MB) 35.3 / 32.9, 4544 -> 13632 31.7 / 28.8, one token 33.1 / 30.0; the projection of 100 tokens 36.4 / 35.0.  The other
// side: one layer's step again and again, its weights then out of that cache, 27.2 / 32.3 and 26.7 / 28.1; and weights of 6 MB,
// of which the caches hold many layers, 11.0 / 13.0.
inline bool weights_stream(const GemmArgs& a) {
    int64_t columns = 0;
    for (int i = 0; i < 3; ++i) columns += a.p[i].n;
    return columns * a.K * 2 >= (int64_t)64 << 20;
}

// 256 x 256 workgroup tiles, for problems large enough to fill the chip with them (prenorm_qkv_wide.hip).
int launch_prenorm_qkv_wide(GemmArgs a, hipStream_t stream);
int64_t prenorm_qkv_wide_tiles(const GemmArgs& a);

// At most 64 tokens: panels of 64 or 32 columns streamed by eight waves that split the contraction (prenorm_qkv_skinny.hip).
int launch_prenorm_qkv_skinny(GemmArgs a, hipStream_t stream);

// 64 x 64, 128 x 64 or 128 x 128 tiles (tokens x columns) whose waves split the contraction, for problems that leave the
// larger tilings with fewer tiles than CUs (prenorm_qkv_mid.hip); the number of such tiles.
int launch_prenorm_qkv_mid(const GemmArgs& a, int mt, int nt, hipStream_t stream);
int64_t prenorm_qkv_mid_tiles(const GemmArgs& a, int mt, int nt);

// The 128 x 128 tiling with two workgroups per CU, and the choice between them all (prenorm_qkv.hip).
int launch_projections(GemmArgs a, hipStream_t stream);

}  // namespace trn
