// Pruned 3D transforms between modes |k| <= h and n >= 2 h points per axis, as
// matrix products of small DFT matrices with the FP64 matrix instructions, one
// axis after the other.
//
// Pairs k and -k (or l and -l) are folded before the product: with
// E = v(k) + v(-k), O = v(k) - v(-k),
//   sum_k v(k) exp(-i t k l) = C - i S,  C = sum_{k >= 0} E cos(t k l),
//                                         S = sum_{k >= 0} O sin(t k l),
// and the output at -l is C + i S: a quarter of the plain matrix product's
// work.  At the sizes in use (h <= 160) that beats an FFT, which moves the
// whole n^3 complex grid through memory once per axis: only the modes and the
// half of the points that symmetry leaves are ever stored.
//
// A workgroup stages the folded values (E, O) of 16 columns in LDS (32 in the
// convolution's middle kernel), all of the contracted axis, and its waves share the
// 16-wide output tiles.  The trigonometric operand comes from a table in memory
// (cos, sin per entry), which stays in L2.
//
// Fine grid of a model, the whole call (FP64 n^3 complex FFT of the padded grid
// before, three kernels now): M = 41 62 -> 21 us, 81 156 -> 41, 121 599 -> 85,
// 162 1,490 -> 200, 320 11,600 -> 2,080; a plan's first model 1.1 s (the FFT
// library's setup) -> 0.5 ms, its buffers (M = 121) 250 -> 46 MB.  Convolution at
// M = 81 on 162^3 points 90 us (FFT pair with its copies 220), M = 121 on 242^3 248.
// Modes of a spread grid (a thread per 8 outputs with a sincos table in LDS before):
// 323 us less 250 at M = 81, 1,520 us less at M = 162.
// Bound: the chain of one workgroup (load, 2 to 40 products, store) more than the
// matrix cores (12 us of the 85 at M = 121) or the 82 MB written.  One column tile
// a workgroup beats two (M = 121 97 against 116 us, M = 41 21 against 30, at four
// waves): more workgroups, at twice the table reads.  A wave per output tile beats
// four waves (M = 121 85 against 99 us, M = 320 2,080 against 2,890, the
// convolution 93 against 113).
#include <algorithm>

#include "nufft_shared.h"

namespace {

typedef double double4v __attribute__((ext_vector_type(4)));

// T[c][o] = (cos, sin)(2 pi c o / n) for contracted index c < nc, output index
// o < no; zero elsewhere (Cp x Op entries).
__global__ __launch_bounds__(256) void k_trig_table(double2 *__restrict__ T, int nc, int Cp,
                                                    int no, int Op, int n)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= Cp * Op) return;
    const int c = i / Op, o = i % Op;
    double s = 0.0, cs = 0.0;
    if (c < nc && o < no) sincospi(2.0 * (double)((c * o) % n) / (double)n, &s, &cs);
    T[i] = make_double2(cs, s);
}

// Stages load(c, col) -> (E, O) for all c < nc and the workgroup's 16 columns into
// s[c * pitch + col]; rows nc .. Cp are zero.  CFAST: consecutive threads take
// consecutive c (the contracted axis is the contiguous one in memory).
template <bool CFAST, class Load>
__device__ __forceinline__ void dft_stage(double2 *s, int pitch, int nc, int Cp, Load load)
{
    if constexpr (CFAST) {
        const int nw = blockDim.x >> 6;
#pragma unroll 4
        for (int col = threadIdx.x >> 6; col < 16; col += nw)
            for (int c = threadIdx.x & 63; c < Cp; c += 64)
                s[c * pitch + col] = c < nc ? load(c, col) : make_double2(0.0, 0.0);
    } else {
        const int col = threadIdx.x & 15, step = blockDim.x >> 4;
#pragma unroll 4
        for (int c = threadIdx.x >> 4; c < Cp; c += step)
            s[c * pitch + col] = c < nc ? load(c, col) : make_double2(0.0, 0.0);
    }
}

// C and S over c in [c0, c1) of the staged columns for the output tiles of 16
// first + step j < count, j < NT = ceil(count / step); a tile past the end is left
// at zero.  Element r of C or S in this lane belongs to column (or output)
// 4 r + lane / 16 and output (or column) lane % 16: with DATA_A the columns are the
// rows of the product and the outputs run along the lanes, otherwise the outputs
// are the rows and the columns run along the lanes.
template <int CT, int NT, bool DATA_A>
__device__ __forceinline__ void dft_tiles(const double2 *s, int pitch, int c0, int c1,
                                          const double2 *__restrict__ T, int Op, int first, int step,
                                          int count, double4v (&C)[NT][CT], double4v (&S)[NT][CT])
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) C[j][ct] = S[j][ct] = double4v{0.0, 0.0, 0.0, 0.0};
    const double2 *t = T + (lane >> 4) * Op + first * 16 + (lane & 15);
    const double2 *d = s + (lane >> 4) * pitch + (lane & 15);
    auto run = [&](auto ntc) __attribute__((always_inline)) {
        constexpr int N = decltype(ntc)::value;
        if constexpr (N > 0) {
#pragma unroll 4
            for (int c = c0; c < c1; c += 4) {
                double2 e[N];
#pragma unroll
                for (int j = 0; j < N; ++j) e[j] = t[c * Op + 16 * step * j];
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) {
                    const double2 v = d[c * pitch + 16 * ct];
#pragma unroll
                    for (int j = 0; j < N; ++j) {
                        const double ax = DATA_A ? v.x : e[j].x, bx = DATA_A ? e[j].x : v.x;
                        const double ay = DATA_A ? v.y : e[j].y, by = DATA_A ? e[j].y : v.y;
                        C[j][ct] = __builtin_amdgcn_mfma_f64_16x16x4f64(ax, bx, C[j][ct], 0, 0, 0);
                        S[j][ct] = __builtin_amdgcn_mfma_f64_16x16x4f64(ay, by, S[j][ct], 0, 0, 0);
                    }
                }
            }
        }
    };
    // every wave has NT or NT - 1 tiles (or none, where there are more waves than tiles)
    if (first + step * (NT - 1) < count) run(std::integral_constant<int, NT>{});
    else run(std::integral_constant<int, NT - 1>{});
}

// All of the contracted axis, output tiles shared by the workgroup's waves.
template <int CT, int NT, bool DATA_A>
__device__ __forceinline__ void dft_all(const double2 *s, int pitch, int Cp,
                                        const double2 *__restrict__ T, int Op, double4v (&C)[NT][CT],
                                        double4v (&S)[NT][CT])
{
    dft_tiles<CT, NT, DATA_A>(s, pitch, 0, Cp, T, Op, __builtin_amdgcn_readfirstlane(threadIdx.x >> 6),
                              blockDim.x >> 6, Op / 16, C, S);
}

__device__ __forceinline__ double shfl_xor1_f64(double v)
{
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0xB1, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0xB1, 0xf, 0xf, false);
    return __hiloint2double(hi, lo);
}

// store(lt, C, S) of the wave's tiles lt (some may lie past the end).
template <int NT, class Store>
__device__ __forceinline__ void for_tiles(const double4v (&C)[NT][1], const double4v (&S)[NT][1],
                                          Store store)
{
#pragma unroll
    for (int j = 0; j < NT; ++j)
        store((int)(threadIdx.x >> 6) + (int)(blockDim.x >> 6) * j, C[j][0], S[j][0]);
}

// ------------------------------------------------- modes -> fine grid (type 2)

// g(k1, k2, k3) of the symmetrised, deconvolved model.
__device__ __forceinline__ double model_mode(const float *__restrict__ ac,
                                             const double *__restrict__ dinv, int M, int h, int k1,
                                             int k2, int k3)
{
    const int lo = -(M / 2), hi = (M - 1) / 2;
    double s = 0.0;
    if (k1 >= lo && k1 <= hi && k2 >= lo && k2 <= hi && k3 >= lo && k3 <= hi)
        s += ac[((int64_t)(k1 + M / 2) * M + (k2 + M / 2)) * M + (k3 + M / 2)];
    if (-k1 >= lo && -k1 <= hi && -k2 >= lo && -k2 <= hi && -k3 >= lo && -k3 <= hi)
        s += ac[((int64_t)(-k1 + M / 2) * M + (-k2 + M / 2)) * M + (-k3 + M / 2)];
    return 0.5 * s * dinv[k1 + h] * dinv[k2 + h] * dinv[k3 + h];
}

// Axis 1: column (k2, k3 >= 0), outputs l1 in [0, n/2]; w1[l1][k2][k3].
template <int NT>
__global__ __launch_bounds__(512) void k_grid_axis1(const float *__restrict__ ac,
                                                    const double *__restrict__ dinv,
                                                    const double2 *__restrict__ T, int Cp, int Op,
                                                    double2 *__restrict__ w1, int M, int h, int n)
{
    extern __shared__ double2 s_dft[];
    const int nh = h + 1, ncol = (2 * h + 1) * nh, col0 = blockIdx.x * 16, lane = threadIdx.x & 63;
    dft_stage<false>(s_dft, 16, nh, Cp, [&](int k1, int j) {
        const int c = col0 + j;
        if (c >= ncol) return make_double2(0.0, 0.0);
        const int k2 = c / nh - h, k3 = c % nh;
        const double a = model_mode(ac, dinv, M, h, k1, k2, k3);
        if (k1 == 0) return make_double2(a, 0.0);
        const double b = model_mode(ac, dinv, M, h, -k1, k2, k3);
        return make_double2(a + b, a - b);
    });
    __syncthreads();
    double4v Cs[NT][1], Ss[NT][1];
    dft_all<1, NT, false>(s_dft, 16, Cp, T, Op, Cs, Ss);
    for_tiles<NT>(Cs, Ss, [&](int lt, double4v C, double4v S) {
        const int c = col0 + (lane & 15);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int l1 = lt * 16 + 4 * r + (lane >> 4);
            if (c < ncol && l1 <= n / 2) w1[(int64_t)l1 * ncol + c] = make_double2(C[r], -S[r]);
        }
    });
}

// Axis 2 of plane l1 (blockIdx.y): column (k3, re / im), outputs l2 in [0, n);
// w2[l1][l2][k3].
template <int NT>
__global__ __launch_bounds__(512) void k_grid_axis2(const double *__restrict__ w1,
                                                    const double2 *__restrict__ T, int Cp, int Op,
                                                    double *__restrict__ w2, int h, int n)
{
    extern __shared__ double2 s_dft[];
    const int nh = h + 1, ncol = 2 * nh, col0 = blockIdx.x * 16, lane = threadIdx.x & 63;
    const double *in = w1 + (int64_t)blockIdx.y * (2 * h + 1) * ncol + (int64_t)h * ncol;
    double *out = w2 + (int64_t)blockIdx.y * n * ncol;
    dft_stage<false>(s_dft, 16, nh, Cp, [&](int k2, int j) {
        const int c = col0 + j;
        if (c >= ncol) return make_double2(0.0, 0.0);
        const double a = in[k2 * ncol + c];
        if (k2 == 0) return make_double2(a, 0.0);
        const double b = in[-k2 * ncol + c];
        return make_double2(a + b, a - b);
    });
    __syncthreads();
    double4v Cs[NT][1], Ss[NT][1];
    dft_all<1, NT, false>(s_dft, 16, Cp, T, Op, Cs, Ss);
    for_tiles<NT>(Cs, Ss, [&](int lt, double4v C, double4v S) {
        const int c = col0 + (lane & 15);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            // C -+ i S: the real part takes +- the imaginary column's S, the
            // imaginary part -+ the real column's
            double o = shfl_xor1_f64(S[r]);
            if (c & 1) o = -o;
            const int l2 = lt * 16 + 4 * r + (lane >> 4);
            if (c < ncol && l2 <= n / 2) {
                out[(int64_t)l2 * ncol + c] = C[r] + o;
                if (l2 > 0 && 2 * l2 != n) out[(int64_t)(n - l2) * ncol + c] = C[r] - o;
            }
        }
    });
}

// Axis 3 of rows (l1 <= n/2, l2): real values at every l3, written as float32 at
// every padded position of (l1, l2, l3) and of (-l1, -l2, -l3), which has the same
// value (the model is even).
template <int NT>
__global__ __launch_bounds__(512) void k_grid_axis3(const double2 *__restrict__ w2,
                                                    const double2 *__restrict__ T, int Cp, int Op,
                                                    float *__restrict__ grid, int h, int n, int np,
                                                    int off)
{
    extern __shared__ double2 s_dft[];
    constexpr int pitch = 17;
    const int nh = h + 1, nrow = (n / 2 + 1) * n, row0 = blockIdx.x * 16;
    const int lane = threadIdx.x & 63;
    dft_stage<true>(s_dft, pitch, nh, Cp, [&](int k3, int j) {
        const int r = row0 + j;
        if (r >= nrow) return make_double2(0.0, 0.0);
        const double2 v = w2[(int64_t)r * nh + k3];
        return k3 == 0 ? make_double2(v.x, 0.0) : make_double2(2.0 * v.x, 2.0 * v.y);
    });
    __syncthreads();
    double4v Cs[NT][1], Ss[NT][1];
    dft_all<1, NT, true>(s_dft, pitch, Cp, T, Op, Cs, Ss);
    __syncthreads();
    // the rows as float32 at their padded positions, over the staged columns
    float *rows = reinterpret_cast<float *>(s_dft);
    const int off0 = off % n;
    // smallest padded position of index l in (-n, n)
    auto first = [&](int l) {
        const int p = l + off0;
        return p < 0 ? p + n : p >= n ? p - n : p;
    };
    for_tiles<NT>(Cs, Ss, [&](int lt, double4v C, double4v S) {
        const int l3 = lt * 16 + (lane & 15);
        if (l3 > n / 2) return;
        const int pa = first(l3), pb = first(-l3);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            float *o = rows + (4 * r + (lane >> 4)) * np;
            const float vp = (float)(C[r] + S[r]), vm = (float)(C[r] - S[r]);
            for (int p = pa; p < np; p += n) o[p] = vp;
            if (pb != pa)
                for (int p = pb; p < np; p += n) o[p] = vm;
        }
    });
    __syncthreads();
    // a wave per row: its copies, and mirrored those of (-l1, -l2); the row's values
    // are read once for all copies
    for (int j = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); j < 16; j += blockDim.x >> 6) {
        const int row = row0 + j;
        if (row >= nrow) break;
        const int l1 = row / n, l2 = row - l1 * n;
        const int images = l1 == 0 || 2 * l1 == n ? 1 : 2;
        for (int im = 0; im < images; ++im)
            for (int q0 = lane; q0 < np; q0 += 256) {
                float v[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    // index -l lies at np - p (2 off = np); np - 0 is a copy of np - n
                    const int p = min(q0 + 64 * u, np - 1);
                    v[u] = rows[j * np + (im ? (p ? np - p : np - n) : p)];
                }
                for (int p1 = first(im ? -l1 : l1); p1 < np; p1 += n)
                    for (int p2 = first(im ? -l2 : l2); p2 < np; p2 += n) {
                        float *o = grid + ((int64_t)p1 * np + p2) * np + q0;
#pragma unroll
                        for (int u = 0; u < 4; ++u)
                            if (q0 + 64 * u < np) o[64 * u] = v[u];
                    }
            }
    }
}

// ---------------------------------- convolution with a kernel given by its spectrum
//
// out = scale s . crop(K * pad(s . u)) + coef base on M^3 values (mtip_merge_conv, for C
// callers; Merge keeps the FFTs' rounding, see adjoint.hip), K cyclic on n^3
// points, n >= M, F its spectrum (l1 in [0, n/2], l2, l3).  Axis 1 and 2 forward,
// then axis 3 forward, the product with F and axis 3 back in one kernel, so the
// full spectrum of u is never stored, then axis 2 and 1 back.  Value i of an axis
// is mode i - M/2 (a cyclic shift, which the convolution commutes with).

// Axis 1: column (i2, i3) of s . u, outputs l1 in [0, n/2]; w1[l1][i2][i3].
template <int NT>
__global__ __launch_bounds__(512) void k_conv_axis1(const double *__restrict__ u,
                                                    const double *__restrict__ sup,
                                                    const double2 *__restrict__ T, int Cp, int Op,
                                                    double2 *__restrict__ w1, int M, int n)
{
    extern __shared__ double2 s_dft[];
    const int h = M / 2, ncol = M * M, col0 = blockIdx.x * 16, lane = threadIdx.x & 63;
    dft_stage<false>(s_dft, 16, h + 1, Cp, [&](int k, int j) {
        const int c = col0 + j;
        if (c >= ncol) return make_double2(0.0, 0.0);
        const int64_t ia = (int64_t)(h + k) * ncol + c, ib = (int64_t)(h - k) * ncol + c;
        const bool in = h + k < M;                 // M even has no mode + M / 2
        double a = in ? u[ia] : 0.0, b = k ? u[ib] : 0.0;
        if (sup) {
            a *= in ? sup[ia] : 0.0;
            b *= k ? sup[ib] : 0.0;
        }
        return make_double2(a + b, a - b);
    });
    __syncthreads();
    double4v Cs[NT][1], Ss[NT][1];
    dft_all<1, NT, false>(s_dft, 16, Cp, T, Op, Cs, Ss);
    for_tiles<NT>(Cs, Ss, [&](int lt, double4v C, double4v S) {
        const int c = col0 + (lane & 15);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int l1 = lt * 16 + 4 * r + (lane >> 4);
            if (c < ncol && l1 <= n / 2) w1[(int64_t)l1 * ncol + c] = make_double2(C[r], -S[r]);
        }
    });
}

// Axis 2 of plane l1 (blockIdx.y): column (i3, re / im).  Forward: M values to n
// points l2.  Back (INV): n points to M values.
template <int NT, bool INV>
__global__ __launch_bounds__(512) void k_conv_axis2(const double *__restrict__ in,
                                                    const double2 *__restrict__ T, int Cp, int Op,
                                                    double *__restrict__ out, int M, int n)
{
    extern __shared__ double2 s_dft[];
    const int h = M / 2, ncol = 2 * M, col0 = blockIdx.x * 16, lane = threadIdx.x & 63;
    const int nin = INV ? n : M, nout = INV ? M : n;
    in += (int64_t)blockIdx.y * nin * ncol;
    out += (int64_t)blockIdx.y * nout * ncol;
    dft_stage<false>(s_dft, 16, (INV ? n / 2 : h) + 1, Cp, [&](int k, int j) {
        const int c = col0 + j;
        if (c >= ncol) return make_double2(0.0, 0.0);
        const int ia = INV ? k : h + k, ib = INV ? n - k : h - k;
        const double a = ia < nin ? in[(int64_t)ia * ncol + c] : 0.0;
        const double b = k > 0 && ib != ia ? in[(int64_t)ib * ncol + c] : 0.0;
        return make_double2(a + b, a - b);
    });
    __syncthreads();
    double4v Cs[NT][1], Ss[NT][1];
    dft_all<1, NT, false>(s_dft, 16, Cp, T, Op, Cs, Ss);
    for_tiles<NT>(Cs, Ss, [&](int lt, double4v C, double4v S) {
        const int c = col0 + (lane & 15);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            // forward C - i S at l2 and C + i S at -l2, back the other way round: the
            // real part takes +- the imaginary column's S, the imaginary part -+ the
            // real column's
            double o = shfl_xor1_f64(S[r]);
            if ((c & 1) != (int)INV) o = -o;
            const int l = lt * 16 + 4 * r + (lane >> 4);
            if (c >= ncol || l > (INV ? h : n / 2)) continue;
            const int ia = INV ? h + l : l, ib = INV ? h - l : n - l;
            if (ia < nout) out[(int64_t)ia * ncol + c] = C[r] + o;
            if (l > 0 && ib != ia) out[(int64_t)ib * ncol + c] = C[r] - o;
        }
    });
}

// Axis 3 of 16 rows (l1, l2), in place: M values to n points, times F, back to M
// values.  Columns 0 - 15 are the rows' real parts, 16 - 31 their imaginary parts.
// The way back has fewer output tiles than waves: the points are split over
// n_split groups of waves, whose sums meet in LDS.
template <int NT, int NI>
__global__ __launch_bounds__(512) void k_conv_axis3(double2 *__restrict__ w2,
                                                    const double2 *__restrict__ F,
                                                    const double2 *__restrict__ T, int Cp, int Op,
                                                    const double2 *__restrict__ Ti, int Cpi,
                                                    int Opi, int n_split, int M, int n)
{
    extern __shared__ double2 s_dft[];
    constexpr int pitch = 33;
    const int h = M / 2, nrow = (n / 2 + 1) * n, row0 = blockIdx.x * 16;
    const int lane = threadIdx.x & 63, l_of = lane & 15, r_of = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nw = blockDim.x >> 6;
#pragma unroll 4
    for (int j = wave; j < 16; j += nw)
        for (int k = lane; k < Cp; k += 64) {
            double2 a = make_double2(0.0, 0.0), b = a;
            if (row0 + j < nrow && k <= h) {
                const double2 *row = w2 + (int64_t)(row0 + j) * M;
                if (h + k < M) a = row[h + k];
                if (k > 0) b = row[h - k];
            }
            s_dft[k * pitch + j] = make_double2(a.x + b.x, a.x - b.x);
            s_dft[k * pitch + 16 + j] = make_double2(a.y + b.y, a.y - b.y);
        }
    __syncthreads();
    {
        double4v C[NT][2], S[NT][2];
        dft_all<2, NT, true>(s_dft, pitch, Cp, T, Op, C, S);
        __syncthreads();
        // Z(+-l) = (C -+ i S) F(+-l), folded again over +-l, in the columns' place
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const int l = (wave + nw * j) * 16 + l_of;
            if (l >= Cpi) continue;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = row0 + 4 * r + r_of;
                double2 e = make_double2(0.0, 0.0), o = e;
                if (row < nrow && l <= n / 2) {
                    const double2 *f = F + (int64_t)row * n;
                    const double2 fa = f[l];
                    const double xr = C[j][0][r] + S[j][1][r], xi = C[j][1][r] - S[j][0][r];
                    e = make_double2(xr * fa.x - xi * fa.y, xr * fa.y + xi * fa.x);
                    if (l > 0 && 2 * l != n) {
                        const double2 fb = f[n - l];
                        const double yr = C[j][0][r] - S[j][1][r], yi = C[j][1][r] + S[j][0][r];
                        const double zr = yr * fb.x - yi * fb.y, zi = yr * fb.y + yi * fb.x;
                        o = make_double2(e.x - zr, e.y - zi);
                        e = make_double2(e.x + zr, e.y + zi);
                    }
                }
                s_dft[l * pitch + 4 * r + r_of] = make_double2(e.x, o.x);
                s_dft[l * pitch + 16 + 4 * r + r_of] = make_double2(e.y, o.y);
            }
        }
    }
    __syncthreads();
    const int n_out = Opi / 16;
    const int part = n_split > 1 ? wave / n_out : 0, first = wave - part * n_out;
    const int per = (Cpi / 4 + n_split - 1) / n_split * 4;
    double4v C[NI][2], S[NI][2];
    dft_tiles<2, NI, true>(s_dft, pitch, part * per, part < n_split ? min(part * per + per, Cpi) : 0, Ti,
                           Opi, first, n_split > 1 ? n_out : nw, n_out, C, S);
    if (n_split > 1) {          // NI = 1
        __syncthreads();
        double4v *sums = reinterpret_cast<double4v *>(s_dft);
        if (part > 0 && part < n_split) {
            double4v *o = sums + ((part - 1) * n_out + first) * 256 + lane;
            o[0] = C[0][0];
            o[64] = C[0][1];
            o[128] = S[0][0];
            o[192] = S[0][1];
        }
        __syncthreads();
        if (part > 0) return;
        for (int q = 1; q < n_split; ++q) {
            const double4v *o = sums + ((q - 1) * n_out + first) * 256 + lane;
            C[0][0] += o[0];
            C[0][1] += o[64];
            S[0][0] += o[128];
            S[0][1] += o[192];
        }
    }
#pragma unroll
    for (int j = 0; j < NI; ++j) {
        const int k = (first + nw * j) * 16 + l_of;
        if (k > h) continue;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = row0 + 4 * r + r_of;
            if (row >= nrow) continue;
            double2 *o = w2 + (int64_t)row * M;
            if (h + k < M) o[h + k] = make_double2(C[j][0][r] - S[j][1][r], C[j][1][r] + S[j][0][r]);
            if (k > 0) o[h - k] = make_double2(C[j][0][r] + S[j][1][r], C[j][1][r] - S[j][0][r]);
        }
    }
}

// Axis 1 back (the half spectrum's other half is its conjugate), then
// out = scale s . y + coef base (base may be out).
template <int NT>
__global__ __launch_bounds__(512) void k_conv_axis1_inv(const double2 *__restrict__ w1,
                                                        const double2 *__restrict__ T, int Cp,
                                                        int Op, const double *__restrict__ sup,
                                                        double scale, double coef,
                                                        const double *base, double *out, int M,
                                                        int n)
{
    extern __shared__ double2 s_dft[];
    const int h = M / 2, ncol = M * M, col0 = blockIdx.x * 16, lane = threadIdx.x & 63;
    dft_stage<false>(s_dft, 16, n / 2 + 1, Cp, [&](int l, int j) {
        const int c = col0 + j;
        if (c >= ncol) return make_double2(0.0, 0.0);
        const double2 v = w1[(int64_t)l * ncol + c];
        const double w = l == 0 || 2 * l == n ? 1.0 : 2.0;
        return make_double2(w * v.x, w * v.y);
    });
    __syncthreads();
    double4v Cs[NT][1], Ss[NT][1];
    dft_all<1, NT, false>(s_dft, 16, Cp, T, Op, Cs, Ss);
    for_tiles<NT>(Cs, Ss, [&](int lt, double4v C, double4v S) {
        const int c = col0 + (lane & 15);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int k = lt * 16 + 4 * r + (lane >> 4);
            if (c >= ncol || k > h) continue;
            auto put = [&](int i1, double y) {
                const int64_t i = (int64_t)i1 * ncol + c;
                y *= scale;
                out[i] = fma(coef, base[i], sup ? sup[i] * y : y);
            };
            if (h + k < M) put(h + k, C[r] - S[r]);
            if (k > 0) put(h - k, C[r] + S[r]);
        }
    });
}

// ----------------------------------------------------- spread grid -> modes (type 1)
//
// F(k) = sum_l v(l) exp(+i t k l) of the real padded grid (np = n + 2 pad points an
// axis, point p at l = p - off, cyclic in n), folded over l and -l; modes k1 >= 0
// only, the others being conjugates.

// Sum of the padded copies of index l (0 <= l < n) of an axis with the given stride.
__device__ __forceinline__ double folded(const double *v, int64_t stride, int l, int n, int np, int off)
{
    double s = 0.0;
    int p = l + off % n;
    for (p = p >= n ? p - n : p; p < np; p += n) s += v[p * stride];
    return s;
}

// Axis 1: column (p2, p3), outputs k1 in [0, h]; w1[k1][p2][p3].
template <int NT>
__global__ __launch_bounds__(512) void k_modes_axis1(const double *__restrict__ acc,
                                                     const double2 *__restrict__ T, int Cp, int Op,
                                                     double2 *__restrict__ w1, int h, int n, int np,
                                                     int off)
{
    extern __shared__ double2 s_dft[];
    const int ncol = np * np, col0 = blockIdx.x * 16, lane = threadIdx.x & 63;
    dft_stage<false>(s_dft, 16, n / 2 + 1, Cp, [&](int l, int j) {
        const int c = col0 + j;
        if (c >= ncol) return make_double2(0.0, 0.0);
        const double a = folded(acc + c, ncol, l, n, np, off);
        const double b = l > 0 && 2 * l != n ? folded(acc + c, ncol, n - l, n, np, off) : 0.0;
        return make_double2(a + b, a - b);
    });
    __syncthreads();
    double4v Cs[NT][1], Ss[NT][1];
    dft_all<1, NT, false>(s_dft, 16, Cp, T, Op, Cs, Ss);
    for_tiles<NT>(Cs, Ss, [&](int lt, double4v C, double4v S) {
        const int c = col0 + (lane & 15);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int k1 = lt * 16 + 4 * r + (lane >> 4);
            if (c < ncol && k1 <= h) w1[(int64_t)k1 * ncol + c] = make_double2(C[r], S[r]);
        }
    });
}

// Axis 2 of plane k1 (blockIdx.y): column (p3, re / im), outputs k2 in [-h, h];
// w2[k1][k2][p3].
template <int NT>
__global__ __launch_bounds__(512) void k_modes_axis2(const double *__restrict__ w1,
                                                     const double2 *__restrict__ T, int Cp, int Op,
                                                     double *__restrict__ w2, int h, int n, int np,
                                                     int off)
{
    extern __shared__ double2 s_dft[];
    const int ncol = 2 * np, col0 = blockIdx.x * 16, lane = threadIdx.x & 63;
    const double *in = w1 + (int64_t)blockIdx.y * np * ncol;
    double *out = w2 + ((int64_t)blockIdx.y * (2 * h + 1) + h) * ncol;
    dft_stage<false>(s_dft, 16, n / 2 + 1, Cp, [&](int l, int j) {
        const int c = col0 + j;
        if (c >= ncol) return make_double2(0.0, 0.0);
        const double a = folded(in + c, ncol, l, n, np, off);
        const double b = l > 0 && 2 * l != n ? folded(in + c, ncol, n - l, n, np, off) : 0.0;
        return make_double2(a + b, a - b);
    });
    __syncthreads();
    double4v Cs[NT][1], Ss[NT][1];
    dft_all<1, NT, false>(s_dft, 16, Cp, T, Op, Cs, Ss);
    for_tiles<NT>(Cs, Ss, [&](int lt, double4v C, double4v S) {
        const int c = col0 + (lane & 15);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            // C +- i S at +-k2: the real part takes -+ the imaginary column's S, the
            // imaginary part +- the real column's
            double o = shfl_xor1_f64(S[r]);
            if (!(c & 1)) o = -o;
            const int k2 = lt * 16 + 4 * r + (lane >> 4);
            if (c >= ncol || k2 > h) continue;
            out[(int64_t)k2 * ncol + c] = C[r] + o;
            if (k2 > 0) out[(int64_t)-k2 * ncol + c] = C[r] - o;
        }
    });
}

// Axis 3 of rows (k1 >= 0, k2), real part, deconvolved: mode (k1, k2, k3) and, for
// k1 > 0, (-k1, -k2, -k3), which has the same real part.
template <int NT>
__global__ __launch_bounds__(512) void k_modes_axis3(const double2 *__restrict__ w2,
                                                     const double2 *__restrict__ T, int Cp, int Op,
                                                     const double *__restrict__ dinv,
                                                     const double *__restrict__ support, double scale,
                                                     double *__restrict__ out, int M, int h, int n,
                                                     int np, int off)
{
    extern __shared__ double2 s_dft[];
    constexpr int pitch = 17;
    const int K = 2 * h + 1, nrow = (h + 1) * K, row0 = blockIdx.x * 16, lane = threadIdx.x & 63;
    dft_stage<true>(s_dft, pitch, n / 2 + 1, Cp, [&](int l, int j) {
        const int r = row0 + j;
        if (r >= nrow) return make_double2(0.0, 0.0);
        const double *v = reinterpret_cast<const double *>(w2 + (int64_t)r * np);
        double e = folded(v, 2, l, n, np, off), o = folded(v + 1, 2, l, n, np, off);
        if (l > 0 && 2 * l != n) {
            e += folded(v, 2, n - l, n, np, off);
            o -= folded(v + 1, 2, n - l, n, np, off);
        }
        return make_double2(e, o);
    });
    __syncthreads();
    double4v Cs[NT][1], Ss[NT][1];
    dft_all<1, NT, true>(s_dft, pitch, Cp, T, Op, Cs, Ss);
    const int lo = -(M / 2), hi = (M - 1) / 2;
    for_tiles<NT>(Cs, Ss, [&](int lt, double4v C, double4v S) {
        const int k = lt * 16 + (lane & 15);
        if (k > h) return;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = row0 + 4 * r + (lane >> 4);
            if (row >= nrow) continue;
            const int k1 = row / K, k2 = row - k1 * K - h;
            auto put = [&](int a, int b, int c, double v) {
                if (a < lo || a > hi || b < lo || b > hi || c < lo || c > hi) return;
                const int64_t i = ((int64_t)(a - lo) * M + (b - lo)) * M + (c - lo);
                out[i] = support ? v * support[i] : v;
            };
            const double w = dinv[k1 + h] * dinv[k2 + h] * dinv[k + h] * scale;
            const double vp = (C[r] - S[r]) * w, vm = (C[r] + S[r]) * w;      // at k3 = k, -k
            put(k1, k2, k, vp);
            if (k > 0) put(k1, k2, -k, vm);
            if (k1 > 0) {
                put(-k1, -k2, -k, vp);
                if (k > 0) put(-k1, -k2, k, vm);
            }
        }
    });
}

int pad_to(int v, int m) { return (v + m - 1) / m * m; }

// Output tiles a wave and waves a workgroup for Op padded outputs: a wave a tile up
// to 8 tiles (M = 81: 6 waves), and at least 4 waves, which also load the columns.
int tiles_a_wave(int Op) { return (Op / 16 + 7) / 8; }
int waves_of(int Op) { return std::max(4, (int)mtip::ceil_div(Op / 16, tiles_a_wave(Op))); }

}  // namespace

namespace mtip {

int grid_from_model(mtip_plan *p, const float *ac, hipStream_t st)
{
    const int h = p->h, n = p->n, nh = h + 1, no = n / 2 + 1;
    const int Cp = pad_to(nh, 4), Op = pad_to(no, 16);
    const size_t n_w1 = (size_t)no * p->K * nh, n_w2 = (size_t)no * n * nh;
    if (!p->G) {
        hipError_t e = hipMalloc(&p->G, (n_w1 + n_w2) * sizeof(double2));
        if (e != hipSuccess) {
            p->G = nullptr;
            return fail(e == hipErrorOutOfMemory ? MTIP_ERR_NOMEM : MTIP_ERR_HIP,
                        std::string("mtip_plan_set_model: ") + hipGetErrorString(e));
        }
    }
    double2 *T = p->gt, *w1 = p->G, *w2 = w1 + n_w1;
    // the staged columns; the padded rows take their place (at most 45 KiB, M = 320)
    const size_t lds = (size_t)Cp * 16 * sizeof(double2);
    const size_t lds3 = std::max((size_t)Cp * 17 * sizeof(double2), (size_t)16 * p->np * sizeof(float));
    const dim3 block(64 * waves_of(Op));
    auto run = [&](auto ntc) {
        constexpr int NT = decltype(ntc)::value;
        hipLaunchKernelGGL((k_grid_axis1<NT>), dim3((unsigned)ceil_div(p->K * nh, 16)), block, lds, st, ac,
                           p->dinv, T, Cp, Op, w1, p->M, h, n);
        hipLaunchKernelGGL((k_grid_axis2<NT>), dim3((unsigned)ceil_div(2 * nh, 16), no), block, lds, st,
                           (const double *)w1, T, Cp, Op, (double *)w2, h, n);
        hipLaunchKernelGGL((k_grid_axis3<NT>), dim3((unsigned)ceil_div((int64_t)no * n, 16)), block, lds3,
                           st, w2, T, Cp, Op, p->grid, h, n, p->np, p->off);
    };
    switch (tiles_a_wave(Op)) {
    case 1: run(std::integral_constant<int, 1>{}); break;
    case 2: run(std::integral_constant<int, 2>{}); break;
    case 3: run(std::integral_constant<int, 3>{}); break;      // n <= 640 (M <= 320)
    default: return fail(MTIP_ERR_ARG, "mtip_plan_set_model: fine grid too large");
    }
    MTIP_HIP_CHECK(hipGetLastError());
    return MTIP_OK;
}

size_t grid_table_entries(const mtip_plan *p)
{
    return (size_t)pad_to(p->h + 1, 4) * pad_to(p->n / 2 + 1, 16);
}

size_t modes_table_entries(const mtip_plan *p)
{
    return (size_t)pad_to(p->n / 2 + 1, 4) * pad_to(p->h + 1, 16);
}

hipError_t trig_tables(const mtip_plan *p)
{
    const int nh = p->h + 1, no = p->n / 2 + 1;
    hipLaunchKernelGGL(k_trig_table, dim3((unsigned)ceil_div(grid_table_entries(p), 256)), dim3(256), 0, 0,
                       p->gt, nh, pad_to(nh, 4), no, pad_to(no, 16), p->n);
    hipLaunchKernelGGL(k_trig_table, dim3((unsigned)ceil_div(modes_table_entries(p), 256)), dim3(256), 0, 0,
                       p->at, no, pad_to(no, 4), nh, pad_to(nh, 16), p->n);
    return hipGetLastError();
}

int modes_from_grid(mtip_plan *p, const double *support, double scale, double *out, hipStream_t st)
{
    const int h = p->h, n = p->n, np = p->np, nh = h + 1;
    const int Cp = pad_to(n / 2 + 1, 4), Op = pad_to(nh, 16);
    const size_t lds = (size_t)Cp * 16 * sizeof(double2), lds3 = (size_t)Cp * 17 * sizeof(double2);
    const dim3 block(64 * waves_of(Op));
    auto run = [&](auto ntc) -> int {
        constexpr int NT = decltype(ntc)::value;
        if (lds3 > 65536)       // M > 237
            for (const void *f : {reinterpret_cast<const void *>(&k_modes_axis1<NT>),
                                  reinterpret_cast<const void *>(&k_modes_axis2<NT>),
                                  reinterpret_cast<const void *>(&k_modes_axis3<NT>)})
                MTIP_HIP_CHECK(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds3));
        hipLaunchKernelGGL((k_modes_axis1<NT>), dim3((unsigned)ceil_div((int64_t)np * np, 16)), block, lds,
                           st, p->acc, p->at, Cp, Op, p->a1, h, n, np, p->off);
        hipLaunchKernelGGL((k_modes_axis2<NT>), dim3((unsigned)ceil_div(2 * np, 16), nh), block, lds, st,
                           (const double *)p->a1, p->at, Cp, Op, (double *)p->a2, h, n, np, p->off);
        hipLaunchKernelGGL((k_modes_axis3<NT>), dim3((unsigned)ceil_div((int64_t)nh * p->K, 16)), block,
                           lds3, st, p->a2, p->at, Cp, Op, p->dinv, support, scale, out, p->M, h, n, np,
                           p->off);
        MTIP_HIP_CHECK(hipGetLastError());
        return MTIP_OK;
    };
    // up to 11 tiles (M <= 320)
    if (tiles_a_wave(Op) == 1) return run(std::integral_constant<int, 1>{});
    return run(std::integral_constant<int, 2>{});
}

}  // namespace mtip

namespace {

// Tables (M values to n points, n points to M values) and the two
// half-transformed arrays of a convolution, in the caller's workspace.
struct ConvLayout {
    int Cp, Op, Cpi, Opi;
    size_t t, ti, w1, w2, total;      // in double2
    ConvLayout(int M, int n)
    {
        const int nh = M / 2 + 1, no = n / 2 + 1;
        Cp = pad_to(nh, 4);
        Op = pad_to(no, 16);
        Cpi = pad_to(no, 4);
        Opi = pad_to(nh, 16);
        t = 0;
        ti = t + (size_t)Cp * Op;
        w1 = ti + (size_t)Cpi * Opi;
        w2 = w1 + (size_t)no * M * M;
        total = w2 + (size_t)no * n * M;
    }
};

bool conv_sizes_ok(int M, int n) { return M >= 2 && n >= M && n <= 320; }

}  // namespace

extern "C" size_t mtip_merge_conv_workspace_size(int M, int M_ups)
{
    return conv_sizes_ok(M, M_ups) ? ConvLayout(M, M_ups).total * sizeof(double2) : 0;
}

extern "C" int mtip_merge_conv_prepare(int M, int M_ups, void *work, size_t work_bytes, void *stream)
{
    MTIP_REQUIRE(conv_sizes_ok(M, M_ups), MTIP_ERR_ARG,
                 "mtip_merge_conv_prepare: need 2 <= M <= M_ups <= 320");
    MTIP_REQUIRE(work, MTIP_ERR_ARG, "mtip_merge_conv_prepare: null pointer");
    const ConvLayout L(M, M_ups);
    MTIP_REQUIRE(work_bytes >= L.total * sizeof(double2), MTIP_ERR_NOMEM,
                 "mtip_merge_conv_prepare: workspace too small");
    double2 *w = (double2 *)work;
    const int nh = M / 2 + 1, no = M_ups / 2 + 1;
    hipStream_t st = (hipStream_t)stream;
    hipLaunchKernelGGL(k_trig_table, dim3((unsigned)mtip::ceil_div(L.Cp * L.Op, 256)), dim3(256), 0, st,
                       w + L.t, nh, L.Cp, no, L.Op, M_ups);
    hipLaunchKernelGGL(k_trig_table, dim3((unsigned)mtip::ceil_div(L.Cpi * L.Opi, 256)), dim3(256), 0,
                       st, w + L.ti, no, L.Cpi, nh, L.Opi, M_ups);
    MTIP_HIP_CHECK(hipGetLastError());
    return MTIP_OK;
}

extern "C" int mtip_merge_conv(const double *u, const double *support, const void *spectrum, int M,
                               int M_ups, double scale, double coef, const double *base, void *work,
                               size_t work_bytes, double *out, void *stream)
{
    MTIP_REQUIRE(conv_sizes_ok(M, M_ups), MTIP_ERR_ARG,
                 "mtip_merge_conv: need 2 <= M <= M_ups <= 320");
    MTIP_REQUIRE(u && spectrum && base && work && out, MTIP_ERR_ARG, "mtip_merge_conv: null pointer");
    MTIP_REQUIRE((uintptr_t)spectrum % 16 == 0 && (uintptr_t)work % 16 == 0, MTIP_ERR_ARG,
                 "mtip_merge_conv: spectrum and workspace must be 16-byte aligned");
    const ConvLayout L(M, M_ups);
    MTIP_REQUIRE(work_bytes >= L.total * sizeof(double2), MTIP_ERR_NOMEM,
                 "mtip_merge_conv: workspace too small");
    const int n = M_ups, no = n / 2 + 1;
    double2 *w = (double2 *)work, *T = w + L.t, *Ti = w + L.ti, *w1 = w + L.w1, *w2 = w + L.w2;
    hipStream_t st = (hipStream_t)stream;
    const size_t lds = (size_t)L.Cp * 16 * sizeof(double2), ldsi = (size_t)L.Cpi * 16 * sizeof(double2);
    const size_t lds3 = (size_t)std::max(L.Cp, L.Cpi) * 33 * sizeof(double2);
    const dim3 cols1((unsigned)mtip::ceil_div((int64_t)M * M, 16));
    const dim3 cols2((unsigned)mtip::ceil_div(2 * M, 16), no);
    const dim3 rows3((unsigned)mtip::ceil_div((int64_t)no * n, 16));
    const double scale_n = scale / ((double)n * n * n);
    const int nw = waves_of(L.Op), n_out = L.Opi / 16;
    // at most a group of waves a tile of points, so the groups' sums (8 KiB a tile) fit
    // where the points' columns were (8.25 KiB a tile)
    const int n_split = std::max(1, std::min(nw, L.Op / 16) / n_out);
    const dim3 block(64 * nw), blocki(64 * waves_of(L.Opi));
    auto run = [&](auto ntc, auto n3c, auto nic) -> int {
        constexpr int NT = decltype(ntc)::value, N3 = decltype(n3c)::value, NI = decltype(nic)::value;
        if (lds3 > 65536)
            MTIP_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_conv_axis3<NT, N3>),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds3));
        hipLaunchKernelGGL((k_conv_axis1<NT>), cols1, block, lds, st, u, support, T, L.Cp, L.Op, w1, M, n);
        hipLaunchKernelGGL((k_conv_axis2<NT, false>), cols2, block, lds, st, (const double *)w1, T, L.Cp,
                           L.Op, (double *)w2, M, n);
        hipLaunchKernelGGL((k_conv_axis3<NT, N3>), rows3, block, lds3, st, w2, (const double2 *)spectrum,
                           T, L.Cp, L.Op, Ti, L.Cpi, L.Opi, n_split, M, n);
        hipLaunchKernelGGL((k_conv_axis2<NI, true>), cols2, blocki, ldsi, st, (const double *)w2, Ti,
                           L.Cpi, L.Opi, (double *)w1, M, n);
        hipLaunchKernelGGL((k_conv_axis1_inv<NI>), cols1, blocki, ldsi, st, w1, Ti, L.Cpi, L.Opi, support,
                           scale_n, coef, base, out, M, n);
        MTIP_HIP_CHECK(hipGetLastError());
        return MTIP_OK;
    };
    // up to 11 tiles of points and of modes; axis 3 has nw waves on the way back too
    const std::integral_constant<int, 1> c1{};
    const std::integral_constant<int, 2> c2{};
    if (tiles_a_wave(L.Op) == 1) return run(c1, c1, c1);
    if (n_out <= nw) return run(c2, c1, c1);
    return tiles_a_wave(L.Opi) == 1 ? run(c2, c2, c1) : run(c2, c2, c2);
}
