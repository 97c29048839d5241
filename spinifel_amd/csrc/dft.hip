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
// A workgroup stages the folded values (E, O) of 16 CT columns in LDS, all of the
// contracted axis, and its four waves share the 16-wide output tiles.  The
// trigonometric operand comes from a table in memory (cos, sin per entry),
// which stays in L2.
//
// Fine grid of a model, the whole call (FP64 n^3 complex FFT of the padded grid
// before, three kernels now): M = 41 62 -> 22 us, 81 156 -> 48, 121 599 -> 99,
// 162 1,490 -> 226, 320 11,600 -> 2,890; a plan's first model 1.1 s (the FFT
// library's setup) -> 0.5 ms, its buffers (M = 121) 250 -> 46 MB.  Bound: the
// chain of one workgroup (load, 2 to 40 products, store) more than the matrix
// cores (12 us of the 99 at M = 121) or the 82 MB written.  One column tile a
// workgroup beats two (M = 121 97 against 116 us, M = 41 21 against 30): more
// workgroups, at twice the table reads.
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

// Stages load(c, col) -> (E, O) for all c < nc and the workgroup's 16 CT columns
// into s[c * pitch + col]; rows nc .. Cp are zero.  CFAST: consecutive threads take
// consecutive c (the contracted axis is the contiguous one in memory).
template <int CT, bool CFAST, class Load>
__device__ __forceinline__ void dft_stage(double2 *s, int pitch, int nc, int Cp, Load load)
{
    constexpr int NCOL = 16 * CT;
    if constexpr (CFAST) {
#pragma unroll 4
        for (int col = threadIdx.x >> 6; col < NCOL; col += 4)
            for (int c = threadIdx.x & 63; c < Cp; c += 64)
                s[c * pitch + col] = c < nc ? load(c, col) : make_double2(0.0, 0.0);
    } else {
        const int col = threadIdx.x % NCOL;
#pragma unroll 4
        for (int c = threadIdx.x / NCOL; c < Cp; c += 256 / NCOL)
            s[c * pitch + col] = c < nc ? load(c, col) : make_double2(0.0, 0.0);
    }
}

// C and S of the staged columns for the wave's output tiles wave + 4 j, j < NT, of
// 16 (a tile past the end is left at zero).  Element r of C or S in this lane
// belongs to column (or output) 4 r + lane / 16 and output (or column) lane % 16:
// with DATA_A the columns are the rows of the product and the outputs run along
// the lanes, otherwise the outputs are the rows and the columns run along the lanes.
template <int CT, int NT, bool DATA_A>
__device__ __forceinline__ void dft_tiles(const double2 *s, int pitch, int Cp,
                                          const double2 *__restrict__ T, int Op,
                                          double4v (&C)[NT][CT], double4v (&S)[NT][CT])
{
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) C[j][ct] = S[j][ct] = double4v{0.0, 0.0, 0.0, 0.0};
    const int last = (Op / 16 - wave + 3) / 4;      // tiles of this wave
    const double2 *t = T + (lane >> 4) * Op + wave * 16 + (lane & 15);
    const double2 *d = s + (lane >> 4) * pitch + (lane & 15);
    auto run = [&](auto ntc) __attribute__((always_inline)) {
        constexpr int N = decltype(ntc)::value;
        if constexpr (N > 0) {
#pragma unroll 4
            for (int c0 = 0; c0 < Cp; c0 += 4) {
                double2 e[N];
#pragma unroll
                for (int j = 0; j < N; ++j) e[j] = t[c0 * Op + 64 * j];
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) {
                    const double2 v = d[c0 * pitch + 16 * ct];
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
    // NT = ceil(tiles / 4): every wave has NT or NT - 1 of them
    if (last >= NT) run(std::integral_constant<int, NT>{});
    else run(std::integral_constant<int, NT - 1>{});
}

__device__ __forceinline__ double shfl_xor1_f64(double v)
{
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0xB1, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0xB1, 0xf, 0xf, false);
    return __hiloint2double(hi, lo);
}

// store(lt, ct, C, S) of the wave's tiles lt (some may lie past the end).
template <int CT, int NT, class Store>
__device__ __forceinline__ void for_tiles(const double4v (&C)[NT][CT], const double4v (&S)[NT][CT],
                                          Store store)
{
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) store((int)(threadIdx.x >> 6) + 4 * j, ct, C[j][ct], S[j][ct]);
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
__global__ __launch_bounds__(256) void k_grid_axis1(const float *__restrict__ ac,
                                                    const double *__restrict__ dinv,
                                                    const double2 *__restrict__ T, int Cp, int Op,
                                                    double2 *__restrict__ w1, int M, int h, int n)
{
    extern __shared__ double2 s_dft[];
    const int nh = h + 1, ncol = (2 * h + 1) * nh, col0 = blockIdx.x * 16, lane = threadIdx.x & 63;
    dft_stage<1, false>(s_dft, 16, nh, Cp, [&](int k1, int j) {
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
    dft_tiles<1, NT, false>(s_dft, 16, Cp, T, Op, Cs, Ss);
    for_tiles<1, NT>(Cs, Ss, [&](int lt, int, double4v C, double4v S) {
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
__global__ __launch_bounds__(256) void k_grid_axis2(const double *__restrict__ w1,
                                                    const double2 *__restrict__ T, int Cp, int Op,
                                                    double *__restrict__ w2, int h, int n)
{
    extern __shared__ double2 s_dft[];
    const int nh = h + 1, ncol = 2 * nh, col0 = blockIdx.x * 16, lane = threadIdx.x & 63;
    const double *in = w1 + (int64_t)blockIdx.y * (2 * h + 1) * ncol + (int64_t)h * ncol;
    double *out = w2 + (int64_t)blockIdx.y * n * ncol;
    dft_stage<1, false>(s_dft, 16, nh, Cp, [&](int k2, int j) {
        const int c = col0 + j;
        if (c >= ncol) return make_double2(0.0, 0.0);
        const double a = in[k2 * ncol + c];
        if (k2 == 0) return make_double2(a, 0.0);
        const double b = in[-k2 * ncol + c];
        return make_double2(a + b, a - b);
    });
    __syncthreads();
    double4v Cs[NT][1], Ss[NT][1];
    dft_tiles<1, NT, false>(s_dft, 16, Cp, T, Op, Cs, Ss);
    for_tiles<1, NT>(Cs, Ss, [&](int lt, int, double4v C, double4v S) {
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
__global__ __launch_bounds__(256) void k_grid_axis3(const double2 *__restrict__ w2,
                                                    const double2 *__restrict__ T, int Cp, int Op,
                                                    float *__restrict__ grid, int h, int n, int np,
                                                    int off)
{
    extern __shared__ double2 s_dft[];
    constexpr int pitch = 17;
    const int nh = h + 1, nrow = (n / 2 + 1) * n, row0 = blockIdx.x * 16;
    const int lane = threadIdx.x & 63;
    dft_stage<1, true>(s_dft, pitch, nh, Cp, [&](int k3, int j) {
        const int r = row0 + j;
        if (r >= nrow) return make_double2(0.0, 0.0);
        const double2 v = w2[(int64_t)r * nh + k3];
        return k3 == 0 ? make_double2(v.x, 0.0) : make_double2(2.0 * v.x, 2.0 * v.y);
    });
    __syncthreads();
    double4v Cs[NT][1], Ss[NT][1];
    dft_tiles<1, NT, true>(s_dft, pitch, Cp, T, Op, Cs, Ss);
    __syncthreads();
    // the rows as float32 at their padded positions, over the staged columns
    float *rows = reinterpret_cast<float *>(s_dft);
    const int off0 = off % n;
    // smallest padded position of index l in (-n, n)
    auto first = [&](int l) {
        const int p = l + off0;
        return p < 0 ? p + n : p >= n ? p - n : p;
    };
    for_tiles<1, NT>(Cs, Ss, [&](int lt, int, double4v C, double4v S) {
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
    for (int j = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); j < 16; j += 4) {
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

int pad_to(int v, int m) { return (v + m - 1) / m * m; }

}  // namespace

namespace mtip {

int grid_from_model(mtip_plan *p, const float *ac, hipStream_t st)
{
    const int h = p->h, n = p->n, nh = h + 1, no = n / 2 + 1;
    const int Cp = pad_to(nh, 4), Op = pad_to(no, 16);
    const size_t n_t = (size_t)Cp * Op, n_w1 = (size_t)no * p->K * nh, n_w2 = (size_t)no * n * nh;
    if (!p->G) {
        hipError_t e = hipMalloc(&p->G, (n_t + n_w1 + n_w2) * sizeof(double2));
        if (e != hipSuccess) {
            p->G = nullptr;
            return fail(e == hipErrorOutOfMemory ? MTIP_ERR_NOMEM : MTIP_ERR_HIP,
                        std::string("mtip_plan_set_model: ") + hipGetErrorString(e));
        }
        hipLaunchKernelGGL(k_trig_table, dim3((unsigned)ceil_div(n_t, 256)), dim3(256), 0, st, p->G,
                           nh, Cp, no, Op, n);
    }
    double2 *T = p->G, *w1 = T + n_t, *w2 = w1 + n_w1;
    // the staged columns; the padded rows take their place (at most 45 KiB, M = 320)
    const size_t lds = (size_t)Cp * 16 * sizeof(double2);
    const size_t lds3 = std::max((size_t)Cp * 17 * sizeof(double2), (size_t)16 * p->np * sizeof(float));
    auto run = [&](auto ntc) {
        constexpr int NT = decltype(ntc)::value;
        hipLaunchKernelGGL((k_grid_axis1<NT>), dim3((unsigned)ceil_div(p->K * nh, 16)),
                           dim3(256), lds, st, ac, p->dinv, T, Cp, Op, w1, p->M, h, n);
        hipLaunchKernelGGL((k_grid_axis2<NT>), dim3((unsigned)ceil_div(2 * nh, 16), no),
                           dim3(256), lds, st, (const double *)w1, T, Cp, Op, (double *)w2, h, n);
        hipLaunchKernelGGL((k_grid_axis3<NT>), dim3((unsigned)ceil_div((int64_t)no * n, 16)),
                           dim3(256), lds3, st, w2, T, Cp, Op, p->grid, h, n, p->np, p->off);
    };
    using std::integral_constant;
    switch ((Op / 16 + 3) / 4) {      // output tiles a wave
    case 1: run(integral_constant<int, 1>{}); break;
    case 2: run(integral_constant<int, 2>{}); break;
    case 3: run(integral_constant<int, 3>{}); break;
    case 4: run(integral_constant<int, 4>{}); break;
    case 5: run(integral_constant<int, 5>{}); break;
    case 6: run(integral_constant<int, 6>{}); break;      // n <= 640 (M <= 320)
    default: return fail(MTIP_ERR_ARG, "mtip_plan_set_model: fine grid too large");
    }
    MTIP_HIP_CHECK(hipGetLastError());
    return MTIP_OK;
}

}  // namespace mtip
