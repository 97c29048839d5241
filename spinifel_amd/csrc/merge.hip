// The merge step's per-iteration vector work on gfx950 (FP64): the operand
// preparation and recombination around the FFTs of
//   W u = support . crop(irfft(rfft(pad(support . u)) . F)) + rlambda u
//         + flambda support . irfft(rfft(support . u) . mask)
// (spinifel/sequential/autocorrelation.py:110-145, :173-178), and the
// conjugate-gradient updates (cupyx/scipy cg, :211-212) with the step
// lengths kept on the device.  Dot products reduce in two fixed-order passes
// (partials per workgroup, then one workgroup), so results do not depend on
// scheduling.
#include "mtip_internal.h"

namespace {

constexpr int kDotBlocks = 512;

// ups[:M, :M, :M] = support . u (the rest of ups stays as the caller zeroed
// it once); us = support . u as an M^3 array for the regulariser's transform.
__global__ __launch_bounds__(256) void k_merge_pad(const double *__restrict__ u,
                                                   const double *__restrict__ s, int M, int Mu,
                                                   double *__restrict__ ups, double *__restrict__ us)
{
    const int64_t n = (int64_t)M * M * M;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int k = (int)(i % M), j = (int)((i / M) % M), l = (int)(i / ((int64_t)M * M));
    const double v = s ? u[i] * s[i] : u[i];
    ups[((int64_t)l * Mu + j) * Mu + k] = v;
    us[i] = v;
}

// out = s . y_ups[:M, :M, :M] + rlambda u + flambda s . y_reg
__global__ __launch_bounds__(256) void k_merge_combine(const double *__restrict__ y_ups,
                                                       const double *__restrict__ y_reg,
                                                       const double *__restrict__ u,
                                                       const double *__restrict__ s, int M,
                                                       int Mu, double rlambda, double flambda,
                                                       double *__restrict__ out)
{
    const int64_t n = (int64_t)M * M * M;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int k = (int)(i % M), j = (int)((i / M) % M), l = (int)(i / ((int64_t)M * M));
    const double sv = s ? s[i] : 1.0;
    const double ada = y_ups[((int64_t)l * Mu + j) * Mu + k] * sv;
    const double fdf = y_reg[i] * sv;
    out[i] = (ada + rlambda * u[i]) + flambda * fdf;
}

__device__ __forceinline__ double block_sum(double v, double *red)
{
    for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m, 64);
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (lane == 0) red[w] = v;
    __syncthreads();
    double t = 0.0;
    if (threadIdx.x == 0)
        for (int i = 0; i < (int)(blockDim.x >> 6); ++i) t += red[i];
    return t;
}

// partial[b] = sum over this workgroup's grid-stride elements of a . b
__global__ __launch_bounds__(256) void k_dot_partial(const double *__restrict__ a,
                                                     const double *__restrict__ b, int64_t n,
                                                     double *__restrict__ partial)
{
    __shared__ double red[4];
    double acc = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        acc = fma(a[i], b[i], acc);
    const double t = block_sum(acc, red);
    if (threadIdx.x == 0) partial[blockIdx.x] = t;
}

__global__ __launch_bounds__(256) void k_dot_final(const double *__restrict__ partial, int n,
                                                   double *__restrict__ out)
{
    __shared__ double red[4];
    double acc = 0.0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) acc += partial[i];
    const double t = block_sum(acc, red);
    if (threadIdx.x == 0) *out = t;
}

// x += (rho / pq) p;  r -= (rho / pq) q
__global__ __launch_bounds__(256) void k_cg_update(double *__restrict__ x, double *__restrict__ r,
                                                   const double *__restrict__ p,
                                                   const double *__restrict__ q,
                                                   const double *__restrict__ rho,
                                                   const double *__restrict__ pq, int64_t n)
{
    const double alpha = *rho / *pq;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        x[i] += alpha * p[i];
        r[i] -= alpha * q[i];
    }
}

// p = r (first) or p = r + (rho / rho_old) p
__global__ __launch_bounds__(256) void k_cg_direction(double *__restrict__ p,
                                                      const double *__restrict__ r,
                                                      const double *__restrict__ rho,
                                                      const double *__restrict__ rho_old,
                                                      int64_t n, int first)
{
    const double beta = first ? 0.0 : *rho / *rho_old;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        p[i] = first ? r[i] : r[i] + beta * p[i];
}

// Half spectrum of M^3 values between its two layouts, M odd: F[i][j][k] with the
// third axis transformed, all of it, and Y[k][i][j], k < M/2 + 1, whose first two axes
// the FFT library then takes contiguous.  Its own real-to-complex path makes the same
// values with one copy more each way and the layouts apart (M = 81: 78 us a pair, 54
// for the four transforms used here).  64 x 16 tiles through LDS.
constexpr int kHalfRows = 64, kHalfCols = 16;

__global__ __launch_bounds__(256) void k_half_pack(const double2 *__restrict__ F, int M,
                                                   double2 *__restrict__ Y)
{
    __shared__ double2 s[kHalfCols][kHalfRows + 1];
    const int h = M / 2 + 1, row0 = blockIdx.x * kHalfRows, k0 = blockIdx.y * kHalfCols;
    const int64_t rows = (int64_t)M * M;
    for (int t = threadIdx.x; t < kHalfRows * kHalfCols; t += 256) {
        const int r = t / kHalfCols, k = t % kHalfCols;
        if (row0 + r < rows && k0 + k < h) s[k][r] = F[(int64_t)(row0 + r) * M + k0 + k];
    }
    __syncthreads();
    for (int t = threadIdx.x; t < kHalfRows * kHalfCols; t += 256) {
        const int r = t % kHalfRows, k = t / kHalfRows;
        if (row0 + r < rows && k0 + k < h) Y[(k0 + k) * rows + row0 + r] = s[k][r];
    }
}

__global__ __launch_bounds__(256) void k_half_expand(const double2 *__restrict__ Y, int M,
                                                     double2 *__restrict__ F)
{
    __shared__ double2 s[kHalfCols][kHalfRows + 1];
    const int h = M / 2 + 1, row0 = blockIdx.x * kHalfRows, k0 = blockIdx.y * kHalfCols;
    const int64_t rows = (int64_t)M * M;
    for (int t = threadIdx.x; t < kHalfRows * kHalfCols; t += 256) {
        const int r = t % kHalfRows, k = t / kHalfRows;
        if (row0 + r < rows && k0 + k < h) s[k][r] = Y[(k0 + k) * rows + row0 + r];
    }
    __syncthreads();
    for (int t = threadIdx.x; t < kHalfRows * kHalfCols; t += 256) {
        const int r = t / kHalfCols, k = k0 + t % kHalfCols;
        if (row0 + r >= rows || k >= h) continue;
        const double2 v = s[k - k0][r];
        double2 *f = F + (int64_t)(row0 + r) * M;
        f[k] = v;
        if (k > 0) f[M - k] = make_double2(v.x, -v.y);
    }
}

// w = (s u, 0)
__global__ __launch_bounds__(256) void k_reg_embed(const double *__restrict__ u,
                                                   const double *__restrict__ s, int64_t n,
                                                   double2 *__restrict__ w)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) w[i] = make_double2(u[i] * s[i], 0.0);
}

// X *= m, m real
__global__ __launch_bounds__(256) void k_reg_mask(double2 *__restrict__ X,
                                                  const double *__restrict__ m, int64_t n)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double2 x = X[i];
    X[i] = make_double2(x.x * m[i], x.y * m[i]);
}

// out += flambda s (scale Re back)
__global__ __launch_bounds__(256) void k_reg_add(const double2 *__restrict__ back, double scale,
                                                 const double *__restrict__ s, double flambda,
                                                 int64_t n, double *__restrict__ out)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] += flambda * (back[i].x * scale) * s[i];
}

// of a launch with a thread a value: it takes fewer than 2^32 threads
constexpr int64_t kMostValues = 256 * (int64_t)0xffffff;

unsigned blocks_for(int64_t n, int64_t cap)
{
    const int64_t b = mtip::ceil_div(n, 256);
    return (unsigned)(b < 1 ? 1 : (b > cap ? cap : b));
}

}  // namespace

extern "C" int mtip_merge_pad(const double *u, const double *support, int M, int M_ups,
                              double *ups, double *us, void *stream)
{
    MTIP_REQUIRE(M >= 1 && M_ups >= M, MTIP_ERR_ARG, "mtip_merge_pad: need 1 <= M <= M_ups");
    MTIP_REQUIRE(u && ups && us, MTIP_ERR_ARG, "mtip_merge_pad: null pointer");
    const int64_t n = (int64_t)M * M * M;
    hipLaunchKernelGGL(k_merge_pad, dim3((unsigned)mtip::ceil_div(n, 256)), dim3(256), 0,
                       (hipStream_t)stream, u, support, M, M_ups, ups, us);
    MTIP_HIP_CHECK(hipGetLastError());
    return MTIP_OK;
}

extern "C" int mtip_merge_combine(const double *y_ups, const double *y_reg, const double *u,
                                  const double *support, int M, int M_ups, double rlambda,
                                  double flambda, double *out, void *stream)
{
    MTIP_REQUIRE(M >= 1 && M_ups >= M, MTIP_ERR_ARG, "mtip_merge_combine: need 1 <= M <= M_ups");
    MTIP_REQUIRE(y_ups && y_reg && u && out, MTIP_ERR_ARG, "mtip_merge_combine: null pointer");
    const int64_t n = (int64_t)M * M * M;
    hipLaunchKernelGGL(k_merge_combine, dim3((unsigned)mtip::ceil_div(n, 256)), dim3(256), 0,
                       (hipStream_t)stream, y_ups, y_reg, u, support, M, M_ups, rlambda, flambda,
                       out);
    MTIP_HIP_CHECK(hipGetLastError());
    return MTIP_OK;
}

extern "C" int mtip_merge_reg_embed(const double *u, const double *support, int64_t n, void *w,
                                    void *stream)
{
    MTIP_REQUIRE(n >= 1 && u && support && w, MTIP_ERR_ARG, "mtip_merge_reg_embed: bad argument");
    MTIP_REQUIRE(n <= kMostValues, MTIP_ERR_ARG, "mtip_merge_reg_embed: too many values");
    hipLaunchKernelGGL(k_reg_embed, dim3((unsigned)mtip::ceil_div(n, 256)), dim3(256), 0,
                       (hipStream_t)stream, u, support, n, (double2 *)w);
    MTIP_HIP_CHECK(hipGetLastError());
    return MTIP_OK;
}

extern "C" int mtip_merge_reg_mask(void *spectrum, const double *mask, int64_t n, void *stream)
{
    MTIP_REQUIRE(n >= 1 && spectrum && mask, MTIP_ERR_ARG, "mtip_merge_reg_mask: bad argument");
    MTIP_REQUIRE(n <= kMostValues, MTIP_ERR_ARG, "mtip_merge_reg_mask: too many values");
    hipLaunchKernelGGL(k_reg_mask, dim3((unsigned)mtip::ceil_div(n, 256)), dim3(256), 0,
                       (hipStream_t)stream, (double2 *)spectrum, mask, n);
    MTIP_HIP_CHECK(hipGetLastError());
    return MTIP_OK;
}

extern "C" int mtip_merge_reg_add(const void *back, double scale, const double *support,
                                  double flambda, int64_t n, double *out, void *stream)
{
    MTIP_REQUIRE(n >= 1 && back && support && out, MTIP_ERR_ARG, "mtip_merge_reg_add: bad argument");
    MTIP_REQUIRE(n <= kMostValues, MTIP_ERR_ARG, "mtip_merge_reg_add: too many values");
    hipLaunchKernelGGL(k_reg_add, dim3((unsigned)mtip::ceil_div(n, 256)), dim3(256), 0,
                       (hipStream_t)stream, (const double2 *)back, scale, support, flambda, n, out);
    MTIP_HIP_CHECK(hipGetLastError());
    return MTIP_OK;
}

extern "C" int mtip_half_pack(const void *spectrum, int M, void *half, void *stream)
{
    MTIP_REQUIRE(M >= 1 && M % 2 == 1 && M <= 2047, MTIP_ERR_ARG, "mtip_half_pack: M must be odd, at most 2047");
    MTIP_REQUIRE(spectrum && half, MTIP_ERR_ARG, "mtip_half_pack: null pointer");
    const dim3 grid((unsigned)mtip::ceil_div((int64_t)M * M, kHalfRows),
                    (unsigned)mtip::ceil_div(M / 2 + 1, kHalfCols));
    hipLaunchKernelGGL(k_half_pack, grid, dim3(256), 0, (hipStream_t)stream, (const double2 *)spectrum, M,
                       (double2 *)half);
    MTIP_HIP_CHECK(hipGetLastError());
    return MTIP_OK;
}

extern "C" int mtip_half_expand(const void *half, int M, void *spectrum, void *stream)
{
    MTIP_REQUIRE(M >= 1 && M % 2 == 1 && M <= 2047, MTIP_ERR_ARG, "mtip_half_expand: M must be odd, at most 2047");
    MTIP_REQUIRE(half && spectrum, MTIP_ERR_ARG, "mtip_half_expand: null pointer");
    const dim3 grid((unsigned)mtip::ceil_div((int64_t)M * M, kHalfRows),
                    (unsigned)mtip::ceil_div(M / 2 + 1, kHalfCols));
    hipLaunchKernelGGL(k_half_expand, grid, dim3(256), 0, (hipStream_t)stream, (const double2 *)half, M,
                       (double2 *)spectrum);
    MTIP_HIP_CHECK(hipGetLastError());
    return MTIP_OK;
}

extern "C" size_t mtip_dot_workspace_size(void) { return kDotBlocks * sizeof(double); }

extern "C" int mtip_dot(const double *a, const double *b, int64_t n, double *work,
                        size_t work_bytes, double *out, void *stream)
{
    MTIP_REQUIRE(n >= 0, MTIP_ERR_ARG, "mtip_dot: n < 0");
    MTIP_REQUIRE(a && b && work && out, MTIP_ERR_ARG, "mtip_dot: null pointer");
    MTIP_REQUIRE(work_bytes >= mtip_dot_workspace_size(), MTIP_ERR_NOMEM,
                 "mtip_dot: workspace smaller than mtip_dot_workspace_size()");
    hipStream_t st = (hipStream_t)stream;
    hipLaunchKernelGGL(k_dot_partial, dim3(kDotBlocks), dim3(256), 0, st, a, b, n, work);
    hipLaunchKernelGGL(k_dot_final, dim3(1), dim3(256), 0, st, work, kDotBlocks, out);
    MTIP_HIP_CHECK(hipGetLastError());
    return MTIP_OK;
}

extern "C" int mtip_cg_update(double *x, double *r, const double *p, const double *q,
                              const double *rho, const double *pq, int64_t n, void *stream)
{
    MTIP_REQUIRE(n >= 0, MTIP_ERR_ARG, "mtip_cg_update: n < 0");
    if (n == 0) return MTIP_OK;
    MTIP_REQUIRE(x && r && p && q && rho && pq, MTIP_ERR_ARG, "mtip_cg_update: null pointer");
    hipLaunchKernelGGL(k_cg_update, dim3(blocks_for(n, 4096)), dim3(256), 0, (hipStream_t)stream,
                       x, r, p, q, rho, pq, n);
    MTIP_HIP_CHECK(hipGetLastError());
    return MTIP_OK;
}

extern "C" int mtip_cg_direction(double *p, const double *r, const double *rho,
                                 const double *rho_old, int64_t n, int first, void *stream)
{
    MTIP_REQUIRE(n >= 0, MTIP_ERR_ARG, "mtip_cg_direction: n < 0");
    if (n == 0) return MTIP_OK;
    MTIP_REQUIRE(p && r && rho && (first || rho_old), MTIP_ERR_ARG,
                 "mtip_cg_direction: null pointer");
    hipLaunchKernelGGL(k_cg_direction, dim3(blocks_for(n, 4096)), dim3(256), 0,
                       (hipStream_t)stream, p, r, rho, rho_old, n, first);
    MTIP_HIP_CHECK(hipGetLastError());
    return MTIP_OK;
}
