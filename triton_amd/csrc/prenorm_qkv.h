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
// of which the last-level cache (256 MB) holds four layers at most and keeps nothing until the same layer comes round again, but would
// evict what it holds for each line.  A trade: a model whose layers come in turn gains, one layer's step again and again on the same
// weights, which then come from HBM each time, loses.  us, whole decode steps, without / with, weights and cache cold (1.4 GB of layers
// in turn); one layer repeated:
//   4096 -> 12288 (96 MB): 1 token on 1024 34.9 / 31.7; 27.2 / 30.0, 16 37.6 / 34.6; 28.3 / 34.0, 32 on 2048 45.0 / 44.1; 33.8 / 40.2, 48 on 1024
//     42.3 / 40.9; 32.6 / 39.2, 64 on 2048 50.0 / 49.3; 38.0 / 47.2, 100 on 4000 67.2 / 67.0; 49.6 / 60.8, 128 on 1024 53.5 / 53.0; 41.0 / 51.0
//   4544 -> 13632 (118 MB): 1 33.9 / 30.2; 27.1 / 28.7, 16 34.6 / 31.0; 27.6 / 30.1, 32 39.8 / 38.9; 31.2 / 34.2, 48 39.0 / 36.1; 30.7 / 35.4, 64 45.7 /
//     44.8; 35.7 / 41.4, 128 58.7 / 56.0; 43.5 / 54.7
//   3584 -> 10752 (73 MB): 1 31.8 / 29.2; 23.8 / 27.1, 16 33.5 / 31.7; 24.9 / 30.4, 64 46.7 / 46.1; 34.0 / 43.0, 128 49.8 / 49.0; 35.3 / 47.0
//   5120 -> 15360 (150 MB): 1 46.6 / 42.3; 35.9 / 40.6, 16 48.4 / 44.7; 36.9 / 43.7, 48 55.0 / 52.2; 40.5 / 50.8, 128 71.0 / 68.7; 51.2 / 67.3
// Below the line a projection alone would go the same way (2816 -> 8448, 45 MB, 16 tokens 15.9 / 15.1; 10.3 / 14.1, 3328 -> 9984, 63 MB 18.5 /
// 17.9; 12.9 / 16.9), but the cache then holds so many layers that a small model's step finds them there.
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

// The checks of trn_linear_f16, and its argument block (not filled in for no tokens).
int linear_args(GemmArgs& a, const void* x, int64_t tokens, int64_t hidden, int64_t ldx, int32_t n_mats, const void* const* w,
                const int64_t* n, const int64_t* ldw, void* const* out, const int64_t* ldo, const void* const* addend);

}  // namespace trn
