// RMSNorm over rows of fp16 data: one pass, the row held in registers between the mean-square
// reduction and the scale.  HBM-bound (few rows: the latency of a row's loads): 16-byte loads, LPR lanes cooperate on one row and reduce
// with cross-lane shuffles, of four waves through LDS; rows*cols*2 bytes read, the same written.
#include <type_traits>
#include "common.h"

namespace trn {

// LPR lanes per row (power of two <= 64, or the workgroup's 256), NV 16-byte vectors per lane.  All of a row's loads are issued before the first is
// waited for (with the squares summed in the same loop the compiler waited for each vector in turn); EARLY: gamma's too.
template <int LPR, int NV, bool EARLY>
__global__ __launch_bounds__(256) void rmsnorm_kernel(
    const half_t* x, const half_t* __restrict__ gamma, half_t* y,     // y may be x (in place): a row is read whole
                                                                     // into registers before any of it is written
    int64_t n_rows, int64_t inner_rows, int cols,
    int64_t x_outer, int64_t ldx, int64_t y_outer, int64_t ldy, int64_t row_start, float eps) {
    constexpr int ROWS_PER_BLOCK = 256 / LPR;
    const int sub = threadIdx.x % LPR;
    const uint32_t row = blockIdx.x * ROWS_PER_BLOCK + threadIdx.x / LPR;
    if (row >= (uint32_t)n_rows) return;             // whole LPR-lane groups leave together
    // 32-bit row arithmetic: the address must be ready before the first load can issue, and a 64-bit
    // division on that path costs more than the whole streaming loop of a short row
    uint32_t outer = 0, inner = row;
    if (inner_rows != n_rows) { outer = row / (uint32_t)inner_rows; inner = row - outer * (uint32_t)inner_rows; }
    const half_t* xr = x + (int64_t)outer * x_outer + ((int64_t)inner + row_start) * ldx;
    half_t* yr = y + (int64_t)outer * y_outer + ((int64_t)inner + row_start) * ldy;

    half8_t v[NV], g[NV];
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int c = (i * LPR + sub) * 8;
        if (c < cols) {
            v[i] = __builtin_nontemporal_load(reinterpret_cast<const half8_t*>(xr + c));   // streamed once: keep it out of the caches' way
            if (EARLY && gamma) g[i] = *reinterpret_cast<const half8_t*>(gamma + c);
        }
    }
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int c = (i * LPR + sub) * 8;
        if (c < cols) {
#pragma unroll
            for (int e = 0; e < 8; ++e) { float f = (float)v[i][e]; ss += f * f; }
        }
    }
#pragma unroll
    for (int m = (LPR < 64 ? LPR : 64) / 2; m >= 1; m >>= 1) ss += __shfl_xor(ss, m, 64);
    if constexpr (LPR == 256) {
        __shared__ float part[4];
        if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = ss;
        __syncthreads();
        ss = (part[0] + part[1]) + (part[2] + part[3]);
    }
    const float rstd = 1.0f / __builtin_sqrtf(ss / (float)cols + eps);

#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int c = (i * LPR + sub) * 8;
        if (c < cols) {
            half8_t o;
            if (gamma) {
                if (!EARLY) g[i] = *reinterpret_cast<const half8_t*>(gamma + c);
#pragma unroll
                for (int e = 0; e < 8; ++e) o[e] = (half_t)((float)g[i][e] * ((float)v[i][e] * rstd));
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) o[e] = (half_t)((float)v[i][e] * rstd);
            }
            __builtin_nontemporal_store(o, reinterpret_cast<half8_t*>(yr + c));
        }
    }
}

template <int LPR, int NV, bool EARLY>
static hipError_t launch_form(const void* x, const void* gamma, void* y, int64_t n_rows, int64_t inner_rows,
                         int cols, int64_t xo, int64_t ldx, int64_t yo, int64_t ldy, int64_t row_start,
                         float eps, hipStream_t s) {
    constexpr int RPB = 256 / LPR;
    dim3 grid((unsigned)((n_rows + RPB - 1) / RPB));
    hipLaunchKernelGGL((rmsnorm_kernel<LPR, NV, EARLY>), grid, dim3(256), 0, s, (const half_t*)x,
                       (const half_t*)gamma, (half_t*)y, n_rows, inner_rows, cols, xo, ldx, yo, ldy,
                       row_start, eps);
    return hipGetLastError();
}

// gamma early or late, of a wave's rows: early is one memory latency instead of two for a row, late leaves the queue to the rows themselves, which
// matters once the resident waves ask for more than the chip takes at a time.  us, before / late / early: 16 x 4096 5.1 / 4.6 /
// 3.9, 396 x 5560 10.4 / 6.7 / 5.4, 300 x 8192 13.3 / 7.9 / 6.2, 1929 x 3216 8.6 / 6.7 / 6.4, 3072 x 4096 11.1 / 9.6 / 8.8, 3400 x
// 4096 11.7 / 10.7 / 12.2, 4096 x 4096 12.8 / 11.4 / 12.5; 1900 x 8192 17.2 / 12.3 / 11.2, 3072 x 6000 17.8 / 14.7 / 14.3, 2500 x
// 8192 19.7 / 16.4 / 18.2; 9000 x 2048 15.9 / 15.8 / 14.5; 12000 x 512 6.8 / 6.8 / 6.5.
// Two vectors a lane: 8192 rows are the waves that the chip holds at once (8 workgroups of 4 rows on each of 256 CUs).  Up to
// there all rows ask at the same moment, and from some 8.5 MB on gamma is better left for later; with more rows the workgroups
// start one by one as others end, and it is not.  late / early: 5000 x 1024 5.06 / 5.06, 7000 x 640 5.25 / 5.31, 7000 x 896 5.78 /
// 6.20, 8192 x 520 5.52 / 5.57, 8192 x 768 5.89 / 6.30, 8192 x 1024 6.96 / 7.90; 8200 x 520 6.45 / 5.96, 8200 x 768 7.46 / 6.78, 8200 x
// 1024 8.36 / 7.87, 12000 x 1016 11.74 / 11.09, 16000 x 1024 14.29 / 13.37; but 2500 x 1024 4.13 / 3.97, 3500 x 520 4.22 / 4.20.
template <int LPR, int NV>
static hipError_t launch(const void* x, const void* gamma, void* y, int64_t n_rows, int64_t inner_rows,
                         int cols, int64_t xo, int64_t ldx, int64_t yo, int64_t ldy, int64_t row_start,
                         float eps, hipStream_t s) {
    auto form = [&](auto early) { return launch_form<LPR, NV, decltype(early)::value>(x, gamma, y, n_rows, inner_rows, cols, xo, ldx, yo, ldy, row_start, eps, s); };
    if constexpr (NV == 1 || NV == 4 || LPR == 256) return form(std::true_type{});
    else if constexpr (NV == 32) return form(std::false_type{});        // (gamma's 32 vectors beside the row's: registers)
    else {
        const int64_t bytes = n_rows * cols * 2;
        const bool early = NV == 2 ? n_rows > 8192 || bytes <= 8500000 : bytes <= (NV == 8 ? 26000000 : 37000000);
        return early ? form(std::true_type{}) : form(std::false_type{});
    }
}

}  // namespace trn

extern "C" int trn_rmsnorm_f16(const void* x, const void* gamma, void* y, int64_t outer_rows,
                               int64_t inner_rows, int64_t cols, int64_t x_outer_stride, int64_t ldx,
                               int64_t y_outer_stride, int64_t ldy, int64_t row_start, float eps,
                               void* stream) {
    using namespace trn;
    if (outer_rows < 0 || inner_rows < 0 || cols <= 0 || row_start < 0) return TRN_E_SHAPE;
    if (outer_rows * inner_rows == 0) return TRN_OK;      // nothing to do; empty tensors have no storage
    if (!x || !y) return TRN_E_NULL;
    if (cols % 8 != 0 || cols > 16384) return TRN_E_SHAPE;
    if (ldx < cols || ldy < cols) return TRN_E_STRIDE;
    if (!aligned16(x) || !aligned16(y) || (gamma && !aligned16(gamma))) return TRN_E_ALIGN;
    if (!pitch16(ldx, 2) || !pitch16(ldy, 2) || !pitch16(x_outer_stride, 2) || !pitch16(y_outer_stride, 2))
        return TRN_E_ALIGN;
    const int64_t n_rows = outer_rows * inner_rows;
    if (n_rows == 0) return TRN_OK;
    if (n_rows > (int64_t)0x7fffffff) return TRN_E_SHAPE;
    hipStream_t s = (hipStream_t)stream;
    const int vecs = (int)(cols / 8);
    hipError_t e;
    // Few long rows: a workgroup has one, whose loads are a quarter as many a lane, instead of four waves one each.  us, wave / workgroup:
    // 1 x 2048 2.60 / 2.22, 64 x 4096 3.88 / 2.59, 1 x 8192 4.68 / 2.91, 200 x 8192 5.89 / 3.99, 64 x 16384 13.2 / 4.2, 400 x 1032 2.97 / 2.95, 400 x 3072 4.44 / 3.34; 1200 x 2048
    // 4.51 / 4.02, 1200 x 4104 6.33 / 5.59, 1200 x 12000 14.3 / 13.7; left out: 800 x 1032 3.18 / 3.24, 2048 x 4096 6.40 / 6.93, 1600 x 8192 9.93 / 10.93, 3000 x 2048 5.39 / 6.32.
    const bool spread = vecs > 128 && n_rows <= (vecs < 160 ? 400 : 1200);
#define TRN_RMS(LPR, NV) e = launch<LPR, NV>(x, gamma, y, n_rows, inner_rows, (int)cols, x_outer_stride, ldx, y_outer_stride, ldy, row_start, eps, s)
    if (vecs <= 8) TRN_RMS(8, 1);
    else if (vecs <= 16) TRN_RMS(16, 1);
    else if (vecs <= 32) TRN_RMS(32, 1);
    else if (vecs <= 64) TRN_RMS(64, 1);
    else if (vecs <= 128) TRN_RMS(64, 2);
    else if (spread && vecs <= 256) TRN_RMS(256, 1);
    else if (spread && vecs <= 512) TRN_RMS(256, 2);
    else if (spread && vecs <= 1024) TRN_RMS(256, 4);
    else if (spread) TRN_RMS(256, 8);
    else if (vecs <= 256) TRN_RMS(64, 4);
    else if (vecs <= 512) TRN_RMS(64, 8);
    else if (vecs <= 1024) TRN_RMS(64, 16);
    else TRN_RMS(64, 32);
#undef TRN_RMS
    return e == hipSuccess ? TRN_OK : TRN_E_LAUNCH;
}
