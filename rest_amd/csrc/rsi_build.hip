// rsi_build.hip — packed B = (μν|Q)·V^{-1/2} written straight into the
// HBM-resident storage of an rjk_ctx (Molecule::prepare_rimatr_for_ri_v_rayon_v02,
// src/molecule_io/mod.rs:1563-1721).
//
//   1. V = (P|Q) on the device (rsi_gpu3c.hip) and V^{-1/2} over its eigenvalues λ > threshold
//      (lapack_power(-0.5, 1e-8), :1582): from a Cholesky factor and its polar factor where every λ
//      is kept, else V's eigenpairs (rocSOLVER dsyevd), W Wᵀ with W = U diag(λ^{-1/4}).
//   2. (μν|Q) in shell-aligned pair slabs, and B[:, slab] = X_slab · V^{-1/2} with one
//      rocBLAS dgemm per slab into the padded [naux][ldb] layout.  Orbital shells beyond d:
//      the slabs come from the host (OpenMP), slab k+1 beside the upload and GEMM of slab k.
//
// Within the workspace limit matrices and slabs live in the context's grow-only workspace and the products use
// its rocBLAS handle, so that a build allocates only what a first build of its size needs.
#include <rocblas/rocblas.h>
#include <rocsolver/rocsolver.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <utility>
#include <vector>

#include "../../include/rest_ri.h"
#include "rjk_internal.hpp"
#include "rsi_gpu3c.hpp"
#include "rsi_internal.hpp"

namespace {

struct Dev {
    void* p = nullptr;
    ~Dev() {
        if (p) (void)hipFree(p);
    }
};
struct Host {
    void* p = nullptr;
    ~Host() {
        if (p) (void)hipHostFree(p);
    }
};
struct Blas {
    rocblas_handle h = nullptr;
    ~Blas() {
        if (h) rocblas_destroy_handle(h);
    }
};
struct GpuInts {
    rsi::Gpu3c g;
    ~GpuInts() { rsi::gpu3c_free(&g); }
};

double now() {
    return std::chrono::duration<double>(std::chrono::steady_clock::now().time_since_epoch()).count();
}

__global__ void k_scale_cols(double* U, int n, const double* w) {
    size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (size_t)n * n) return;
    U[t] *= w[t / n];   // column t / n (column-major)
}

// ---- V^{-1/2} without an eigenproblem ------------------------------------------------
// V = L Lᵀ by Cholesky with the largest remaining diagonal as pivot; the polar factor Q of Lᵀ by scaled
// Newton–Schulz steps X ← X (a − b XᵀX) (Higham, Functions of Matrices, ch. 8); then Lᵀ = Q V^{1/2}
// and V^{-1/2} = L^{-T} Q.  Singular values of Lᵀ are the square roots of V's eigenvalues, and pivoting
// grades its rows, which every step's product on the right keeps.  Against integrals and root in 80 bits B of
// 1 to 3 waters errs by 0.2 to 0.8e-12 of its norm; from rocSOLVER's eigenpairs of the host's V, as before, by 0.7 to
// 1.7e-12 (V's own rounding is most of it; an unpivoted factor adds 1 to 7e-11).  1356 auxiliary functions: 9.3 ms against 31 with dsyevd, whose tridiagonal reduction
// is five dependent launches a column; 113: 1.2 against 2.4; 3164: 75 against 283.  Of the 9.3 ms the
// pivots take 3.5, the 19 steps' products 4.0 (47 TFLOP/s), the updates 0.9, the triangular solve 0.5.
constexpr int kMetBlock = 64;      // pivots between updates of the whole remainder
constexpr int kMetRows = 64;       // rows of a work-group in one pivot's step
constexpr double kMetCut = 1e-13;  // smallest pivot relative to the largest (a pivot up to thr ends it too: V's least eigenvalue is no larger)
constexpr int kMetParts = 1024;    // partial results of a reduction

__global__ __launch_bounds__(256) void k_met_rowsum(const double* __restrict__ V, int n, double* __restrict__ out,
                                                    double* __restrict__ diag, int* __restrict__ state) {
    __shared__ double red[4];
    const int j = blockIdx.x;
    double s = 0.0;
    for (int i = threadIdx.x; i < n; i += 256) s += fabs(V[(size_t)j * n + i]);
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x) return;
    out[j] = (red[0] + red[1]) + (red[2] + red[3]);
    diag[j] = V[(size_t)j * n + j];
    if (j < 2) state[j] = -2;
    if (n == 1) state[1] = -2;
}

// Pivot k, the block's first being k0: S holds V less the blocks before.  Every work-group finds the pivot in
// diag[k % 2] by itself (NaN marks a row that has been one) and writes its rows' diagonals to the other
// half; state[k % 2] is what launch k finds: −2 running, else stopped at that rank.
__global__ __launch_bounds__(256) void k_met_pivot(const double* __restrict__ S, int n, int k, int k0, double thr,
                                                   double* __restrict__ diag, double* __restrict__ top0,
                                                   double* __restrict__ L, int* __restrict__ piv,
                                                   int* __restrict__ state) {
    __shared__ double wmax[4], part[256], lp[kMetBlock];
    __shared__ int widx[4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (state[k & 1] != -2) {   // stopped in an earlier launch (uniform)
        if (blockIdx.x == 0 && tid == 0) state[(k + 1) & 1] = state[k & 1];
        return;
    }
    const double* __restrict__ din = diag + (size_t)(k & 1) * n;
    double mx = -INFINITY;
    int at = 0;
    for (int i = tid; i < n; i += 256) {
        const double d = din[i];
        if (d > mx) {
            mx = d;
            at = i;
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const double m2 = __shfl_xor(mx, o, 64);
        const int a2 = __shfl_xor(at, o, 64);
        if (m2 > mx || (m2 == mx && a2 < at)) {
            mx = m2;
            at = a2;
        }
    }
    if (lane == 0) {
        wmax[wave] = mx;
        widx[wave] = at;
    }
    __syncthreads();
    double top = wmax[0];
    int p = widx[0];
    for (int w = 1; w < 4; ++w)
        if (wmax[w] > top || (wmax[w] == top && widx[w] < p)) {
            top = wmax[w];
            p = widx[w];
        }
    const double d0 = k == 0 ? top : top0[0];
    const bool stop = !(top > kMetCut * d0 && top > thr) || !(top < INFINITY);
    if (blockIdx.x == 0 && tid == 0) {
        if (k == 0) top0[0] = top;
        piv[k] = p;
        state[(k + 1) & 1] = stop ? k : -2;
    }
    if (stop) return;   // uniform over the grid
    if (tid < k - k0) lp[tid] = L[(size_t)(k0 + tid) * n + p];
    __syncthreads();
    const int i = blockIdx.x * kMetRows + lane, nb = k - k0;
    double v = 0.0;
    if (i < n) {
        const double* __restrict__ li = L + (size_t)k0 * n + i;
        double x[kMetBlock / 4];
#pragma unroll
        for (int u = 0; u < kMetBlock / 4; ++u) x[u] = wave + 4 * u < nb ? li[(size_t)(wave + 4 * u) * n] : 0.0;
#pragma unroll
        for (int u = 0; u < kMetBlock / 4; ++u)
            if (wave + 4 * u < nb) v += x[u] * lp[wave + 4 * u];
    }
    part[tid] = v;
    __syncthreads();
    if (wave == 0 && i < n) {
        v = (part[lane] + part[lane + 64]) + (part[lane + 128] + part[lane + 192]);
        const double d = din[i], r = sqrt(top);
        const double l = i == p ? r : (d == d ? (S[(size_t)p * n + i] - v) / r : 0.0);
        L[(size_t)k * n + i] = l;
        diag[(size_t)((k + 1) & 1) * n + i] = i == p ? NAN : d - l * l;
    }
}

// The block's kb <= kMetPanel pivots from k0 in one launch of one work-group, for n <= 1024·kMetOwn: a thread owns
// rows tid + 1024 r and keeps their panel elements in registers; a pivot costs two barriers and one
// column of S.  1356 functions: 2.6 us a pivot against 6.3 for a launch each.  Diagonals in
// diag[0 .. n) throughout; state as launch 0 of the kernel above finds it.
constexpr int kMetOwn = 2, kMetPanel = 16;
template <class F, int... U>
__device__ __forceinline__ void steps(const F& f, std::integer_sequence<int, U...>) {
    (void)(f(std::integral_constant<int, U>()) && ...);   // in order, until one says no; u a constant in each
}
__global__ __launch_bounds__(1024) void k_met_panel(const double* __restrict__ S, int n, int k0, int kb, double thr,
                                                    double* __restrict__ diag, double* __restrict__ top0,
                                                    double* __restrict__ L, int* __restrict__ piv,
                                                    int* __restrict__ state) {
    __shared__ double wmax[2][16], lp[2][kMetPanel];
    __shared__ int widx[2][16];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (state[0] != -2) return;   // stopped in an earlier launch (uniform)
    double l[kMetOwn][kMetPanel], d[kMetOwn];
#pragma unroll
    for (int r = 0; r < kMetOwn; ++r) {
        const int i = tid + 1024 * r;
        d[r] = i < n ? diag[i] : NAN;
    }
    double d0 = k0 ? top0[0] : 0.0;
    const auto step = [&](auto uc) -> bool {   // pivot k0 + u; false: no more
        constexpr int u = decltype(uc)::value;
        if (u >= kb) return false;
        double mx = -INFINITY;
        int p = n;
#pragma unroll
        for (int r = 0; r < kMetOwn; ++r)
            if (d[r] > mx) {
                mx = d[r];
                p = tid + 1024 * r;
            }
        auto best = [&](int o) {
            const double m2 = __shfl_xor(mx, o, 64);
            const int p2 = __shfl_xor(p, o, 64);
            if (m2 > mx || (m2 == mx && p2 < p)) {
                mx = m2;
                p = p2;
            }
        };
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) best(o);
        if (lane == 0) {
            wmax[u & 1][wave] = mx;
            widx[u & 1][wave] = p;
        }
        __syncthreads();
        mx = wmax[u & 1][lane & 15];
        p = widx[u & 1][lane & 15];
#pragma unroll
        for (int o = 8; o > 0; o >>= 1) best(o);
        if (k0 + u == 0) {
            d0 = mx;
            if (tid == 0) top0[0] = mx;
        }
        if (!(mx > kMetCut * d0 && mx > thr) || !(mx < INFINITY)) {   // uniform over the work-group
            if (tid == 0) state[0] = k0 + u;
            return false;
        }
        double s[kMetOwn];
#pragma unroll
        for (int r = 0; r < kMetOwn; ++r) {
            const int i = tid + 1024 * r;
            s[r] = i < n ? S[(size_t)p * n + i] : 0.0;
            if (i == p)
#pragma unroll
                for (int j = 0; j < u; ++j) lp[u & 1][j] = l[r][j];
        }
        if (tid == 0) piv[k0 + u] = p;
        __syncthreads();
        const double root = sqrt(mx);
#pragma unroll
        for (int r = 0; r < kMetOwn; ++r) {
            const int i = tid + 1024 * r;
            double v = s[r];
#pragma unroll
            for (int j = 0; j < u; ++j) v -= l[r][j] * lp[u & 1][j];
            l[r][u] = i == p ? root : (d[r] == d[r] ? v / root : 0.0);
            d[r] = i == p ? NAN : d[r] - l[r][u] * l[r][u];
            if (i < n) L[(size_t)(k0 + u) * n + i] = l[r][u];
        }
        return true;
    };
    steps(step, std::make_integer_sequence<int, kMetPanel>());
#pragma unroll
    for (int r = 0; r < kMetOwn; ++r)
        if (tid + 1024 * r < n) diag[tid + 1024 * r] = d[r];
}

// X0 = s Lᵀ and the triangle Lt[r][c] = L[piv r][c], both column-major; 32 × 32 blocks
__global__ __launch_bounds__(256) void k_met_start(const double* __restrict__ L, int n, const int* __restrict__ piv,
                                                   double s, double* __restrict__ X, double* __restrict__ Lt) {
    __shared__ double t[32][33];
    const int i0 = blockIdx.x * 32, k0 = blockIdx.y * 32, x = threadIdx.x & 31;
    for (int y = threadIdx.x >> 5; y < 32; y += 8) {
        const int i = i0 + x, k = k0 + y;
        if (i < n && k < n) {
            t[y][x] = s * L[(size_t)k * n + i];
            Lt[(size_t)k * n + i] = i < k ? 0.0 : L[(size_t)k * n + piv[i]];
        }
    }
    __syncthreads();
    for (int y = threadIdx.x >> 5; y < 32; y += 8) {
        const int i = i0 + y, k = k0 + x;
        if (i < n && k < n) X[(size_t)i * n + k] = t[x][y];
    }
}

// G ← a I − b G; part: maxima of |G − I| before
__global__ __launch_bounds__(256) void k_met_step(double* __restrict__ G, int n, double a, double b,
                                                  double* __restrict__ part) {
    __shared__ double red[4];
    double m = 0.0;
    for (size_t t = (size_t)blockIdx.x * 256 + threadIdx.x; t < (size_t)n * n; t += (size_t)gridDim.x * 256) {
        const bool d = t / n == t % n;
        const double g = G[t], e = fabs(g - (d ? 1.0 : 0.0));
        m = rjk::max_nan(m, e);
        G[t] = (d ? a : 0.0) - b * g;
    }
    for (int o = 32; o > 0; o >>= 1) m = rjk::max_nan(m, __shfl_xor(m, o, 64));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 4; ++w) m = rjk::max_nan(m, red[w]);
        part[blockIdx.x] = m;
    }
}

// Vm[piv k][c] = Y[k][c]; part: sums of squares
__global__ __launch_bounds__(256) void k_met_rows(const double* __restrict__ Y, int n, const int* __restrict__ piv,
                                                  double* __restrict__ Vm, double* __restrict__ part) {
    __shared__ double red[4];
    double s = 0.0;
    for (size_t t = (size_t)blockIdx.x * 256 + threadIdx.x; t < (size_t)n * n; t += (size_t)gridDim.x * 256) {
        const double y = Y[t];
        Vm[t / n * n + piv[t % n]] = y;
        s += y * y;
    }
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) part[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}

}  // namespace

#define RSI_HIP(ctx, call)                                                                     \
    do {                                                                                       \
        hipError_t e_ = (call);                                                                \
        if (e_ != hipSuccess) {                                                                \
            rsi::set_error(std::string(#call) + ": " + hipGetErrorString(e_));                 \
            return rjk::fail((ctx), RJK_ERR_HIP, std::string(#call) + ": " + hipGetErrorString(e_)); \
        }                                                                                      \
    } while (0)
#define RSI_BLAS(ctx, call)                                                        \
    do {                                                                           \
        rocblas_status s_ = (call);                                                \
        if (s_ != rocblas_status_success) {                                        \
            rsi::set_error(std::string(#call) + " failed: " + std::to_string((int)s_)); \
            return rjk::fail((ctx), RJK_ERR_HIP, std::string(#call) + " failed");  \
        }                                                                          \
    } while (0)

namespace {

// bytes of metric_polar's scratch: [S | L | X | X' | 2 diag | parts | piv | state]
size_t metric_bytes(size_t n) {
    return 4 * rjk::round_up(n * n * sizeof(double), 256) + rjk::round_up((2 * n + 2 * kMetParts + n + 8) * sizeof(double), 256);
}

// Vm = V^{-1/2} where every eigenvalue of V exceeds thr and the steps converge (*done); V is kept.
int metric_polar(rjk_ctx* ctx, rocblas_handle h, hipStream_t st, size_t n, double thr, const double* V, void* scratch,
                 double* Vm, bool* done) {
    *done = false;
    const size_t nn = rjk::round_up(n * n * sizeof(double), 256);
    char* base = (char*)scratch;
    double *S = (double*)base, *L = (double*)(base + nn), *X = (double*)(base + 2 * nn), *X2 = (double*)(base + 3 * nn);
    double* diag = (double*)(base + 4 * nn);
    double* part = diag + 2 * n;               // [2][kMetParts]
    double* top0 = part + 2 * kMetParts;       // the first pivot; the row sums are in X until the steps
    int* state = (int*)(top0 + 2);
    int* piv = state + 2;
    const rocblas_int ni = (rocblas_int)n;
    const double one = 1.0, zero = 0.0, minus = -1.0;
    const unsigned nb = (unsigned)((n + 31) / 32), parts = (unsigned)std::min<size_t>((n * n + 255) / 256, kMetParts);

    RSI_HIP(ctx, rjk::launch_copy(st, S, V, n * n * sizeof(double)));
    hipLaunchKernelGGL(k_met_rowsum, dim3((unsigned)n), dim3(256), 0, st, V, (int)n, X, diag, state);
    const bool panel = n <= 1024 * kMetOwn;
    const size_t block = panel ? kMetPanel : kMetBlock;
    for (size_t k0 = 0; k0 < n; k0 += block) {
        const size_t k1 = std::min(n, k0 + block);
        if (panel)
            hipLaunchKernelGGL(k_met_panel, dim3(1), dim3(1024), 0, st, S, (int)n, (int)k0, (int)(k1 - k0), thr, diag, top0, L, piv,
                               state);
        for (size_t k = panel ? k1 : k0; k < k1; ++k)
            hipLaunchKernelGGL(k_met_pivot, dim3((unsigned)((n + kMetRows - 1) / kMetRows)), dim3(256), 0, st, S, (int)n, (int)k,
                               (int)k0, thr, diag, top0, L, piv, state);
        if (k1 < n)
            RSI_BLAS(ctx, rocblas_dgemm(h, rocblas_operation_none, rocblas_operation_transpose, ni, ni,
                                        (rocblas_int)(k1 - k0), &minus, L + k0 * n, ni, L + k0 * n, ni, &one, S, ni));
    }
    RSI_HIP(ctx, hipGetLastError());
    std::vector<double> sums(n);
    int st2[2] = {0, 0};
    RSI_HIP(ctx, hipMemcpyAsync(sums.data(), X, n * sizeof(double), hipMemcpyDeviceToHost, st));
    RSI_HIP(ctx, hipMemcpyAsync(st2, state, sizeof(st2), hipMemcpyDeviceToHost, st));
    RSI_HIP(ctx, hipStreamSynchronize(st));
    double lam = 0.0;                          // bound of V's eigenvalues
    for (double v : sums) lam = std::max(lam, v);
    if (st2[panel ? 0 : n & 1] != -2 || !(lam > 0.0) || !std::isfinite(lam)) return RJK_OK;

    // Lᵀ/√lam: singular values in [√(thr/lam), 1].  While the lower bound l is small, the cubic that is
    // closest to one on [l, 1] (its extreme values scaled to one); from 0.9 on the plain step.
    hipLaunchKernelGGL(k_met_start, dim3(nb, nb), dim3(256), 0, st, L, (int)n, piv, 1.0 / std::sqrt(lam), X, S);   // S = Lt
    double l = std::max(std::sqrt(std::max(thr, 0.0) / lam), 1e-8);
    double* G = L;                             // L is in S now
    double *x = X, *y = X2;
    for (int it = 0; it < 64; ++it) {
        const bool last = 1.0 - l < 1e-9;      // after this step 1 − l is below rounding
        double a = 1.5, b = 0.5;
        if (l < 0.9) {
            const double q = 1.0 + l + l * l, m = 2.0 / 3.0 * q * std::sqrt(q / 3.0);
            a = q / m;
            b = 1.0 / m;
            l = (q - 1.0) / m;
        } else {
            l = 1.5 * l - 0.5 * l * l * l;
        }
        RSI_BLAS(ctx, rocblas_dgemm(h, rocblas_operation_transpose, rocblas_operation_none, ni, ni, ni, &one, x, ni, x, ni,
                                    &zero, G, ni));
        hipLaunchKernelGGL(k_met_step, dim3(parts), dim3(256), 0, st, G, (int)n, a, b, part);
        RSI_BLAS(ctx, rocblas_dgemm(h, rocblas_operation_none, rocblas_operation_none, ni, ni, ni, &one, x, ni, G, ni, &zero,
                                    y, ni));
        std::swap(x, y);
        if (last) break;
    }
    RSI_BLAS(ctx, rocblas_dtrsm(h, rocblas_side_left, rocblas_fill_lower, rocblas_operation_transpose,
                                rocblas_diagonal_non_unit, ni, ni, &one, S, ni, x, ni));
    hipLaunchKernelGGL(k_met_rows, dim3(parts), dim3(256), 0, st, x, (int)n, piv, Vm, part + kMetParts);
    RSI_HIP(ctx, hipGetLastError());
    std::vector<double> pt(2 * kMetParts);
    RSI_HIP(ctx, hipMemcpyAsync(pt.data(), part, pt.size() * sizeof(double), hipMemcpyDeviceToHost, st));
    RSI_HIP(ctx, hipStreamSynchronize(st));
    double dev = 0.0, norm2 = 0.0;
    for (unsigned k = 0; k < parts; ++k) {
        dev = rjk::max_nan(dev, pt[k]);        // of the last step's XᵀX from one
        norm2 += pt[kMetParts + k];
    }
    // 1/‖V^{-1/2}‖² is at most V's smallest eigenvalue: above thr, the eigenpairs would all be kept
    *done = dev < 1e-8 && 1.0 / norm2 > thr * (1.0 + 1e-6) && norm2 > 0.0;
    return RJK_OK;
}

}  // namespace

extern "C" int rsi_build_rimatr(rjk_ctx* ctx, const rsi_basis* orb, const rsi_basis* aux, double thr,
                                unsigned store_mask, size_t* nkept, double* seconds) {
    if (!ctx || !orb || !aux) {
        rsi::set_error("rsi_build_rimatr: NULL argument");
        return RJK_ERR_ARG;
    }
    if (orb->nbf != ctx->nbf || aux->nbf != ctx->naux) {
        rsi::set_error("rsi_build_rimatr: basis sizes do not match the context");
        return rjk::fail(ctx, RJK_ERR_ARG, "rsi_build_rimatr: basis sizes (" + std::to_string(orb->nbf) + ", " +
                                               std::to_string(aux->nbf) + ") do not match the context");
    }
    const size_t nbf = ctx->nbf, naux = ctx->naux, ldb = ctx->ldb;
    const hipStream_t st = ctx->stream;
    double t_3c = 0, t_v = 0, t_gemm = 0;
    RSI_HIP(ctx, hipSetDevice(ctx->device));
    int rc = rjk::alloc_b(ctx, store_mask);
    if (rc) return rc;
    rocblas_handle h = nullptr;
    rc = rjk::solver_handle(ctx, &h);
    if (rc) return rc;

    // ---- slabs of pair columns j, shell aligned, ≈ 256 MiB of (μν|Q) each --------
    std::vector<size_t> cuts{0};
    {
        const size_t budget = (size_t(256) << 20) / (naux * sizeof(double));   // pairs per slab
        size_t j0 = 0;
        for (const rsi::Shell& s : orb->sh) {
            const size_t jend = s.off + s.nsph;
            if (jend * (jend + 1) / 2 - j0 * (j0 + 1) / 2 > budget && (size_t)s.off > j0) {
                cuts.push_back(s.off);
                j0 = s.off;
            }
        }
        cuts.push_back(nbf);
    }
    size_t maxq = 0;
    for (size_t k = 0; k + 1 < cuts.size(); ++k)
        maxq = std::max(maxq, cuts[k + 1] * (cuts[k + 1] + 1) / 2 - cuts[k] * (cuts[k] + 1) / 2);
    const bool dev3 = rsi::gpu3c_supported(*orb, *aux), dev2 = rsi::gpu3c_aux_supported(*aux);
    GpuInts g;
    if (dev2) {
        const int r = rsi::gpu3c_init(&g.g, dev3 ? orb : nullptr, *aux, dev3 ? cuts : std::vector<size_t>(), st);
        if (r) return rjk::fail(ctx, r, "rsi_build_rimatr: device integral set-up failed");
    }
    // Matrices: U; V^{-1/2} with λ, E, w and info behind it; the metric's scratch, then the X slab of the device
    // route.  Within the workspace limit they are the context's workspace, which the next build finds again.
    // Beyond it, or where that much memory is not to be had, each is an allocation of its own for as
    // long as it is needed, and without room for the metric's scratch the eigenpairs serve.
    const size_t nn = rjk::round_up(naux * naux * sizeof(double), 256), nv = rjk::round_up(naux * sizeof(double), 256);
    const size_t vbytes = nn + 3 * nv + 256, xbytes = dev3 ? maxq * naux * sizeof(double) : 0;
    const size_t need = nn + vbytes + std::max(metric_bytes(naux), xbytes);
    Dev tU, tV, tS, tX;
    const auto temp = [](Dev& d, size_t bytes) {
        if (hipMalloc(&d.p, bytes) == hipSuccess) return true;
        (void)hipGetLastError();
        d.p = nullptr;
        return false;
    };
    void *ws = nullptr, *dU_ = nullptr, *dV_ = nullptr, *dS = nullptr, *dX_ = nullptr;
    const std::string err = ctx->err;
    if (need <= std::max(ctx->ws_limit, ctx->ws_size) && rjk::ws_get(ctx, need, &ws) == RJK_OK) {
        dU_ = ws;
        dV_ = (char*)ws + nn;
        dS = dX_ = (char*)dV_ + vbytes;
    } else {
        ctx->err = err;
        if (!temp(tU, nn) || !temp(tV, vbytes))
            return rjk::fail(ctx, RJK_ERR_NOMEM, "rsi_build_rimatr: device allocation of the metric failed");
        (void)temp(tS, metric_bytes(naux));
        dU_ = tU.p;
        dV_ = tV.p;
        dS = tS.p;
    }
    double* dU = (double*)dU_;
    double* dVm = (double*)dV_;
    double* dlam = (double*)((char*)dV_ + nn);
    double* dE = (double*)((char*)dlam + nv);
    double* dw = (double*)((char*)dE + nv);
    rocblas_int* dinfo = (rocblas_int*)((char*)dw + nv);

    // ---- V^{-1/2} ----------------------------------------------------------
    double t0 = now();
    if (dev2) {
        if (rsi::gpu2c(g.g, st, dU, naux))
            return rjk::fail(ctx, RJK_ERR_HIP, "rsi_build_rimatr: two-centre kernel launch failed");
    } else {
        std::vector<double> V(naux * naux);
        rc = rsi_int2c2e(aux, V.data());
        if (rc) return rjk::fail(ctx, rc, rsi::last_error());
        RSI_HIP(ctx, hipMemcpyAsync(dU, V.data(), naux * naux * sizeof(double), hipMemcpyHostToDevice, st));
        RSI_HIP(ctx, hipStreamSynchronize(st));
    }
    size_t kept = naux;
    bool polar = false;
    if (dS) rc = metric_polar(ctx, h, st, naux, thr, dU, dS, dVm, &polar);
    if (rc) return rc;
    ++ctx->routes[polar ? RJK_ROUTE_METRIC_POLAR : RJK_ROUTE_METRIC_EIGENPAIRS];
    if (tS.p) (void)hipFree(std::exchange(tS.p, nullptr));
    if (!polar) {
        // the eigensolver's workspace, a few matrices, stays with its handle: a large one gets a handle of its own (up
        // to 2147 functions the 128 MiB that any handle holds are enough; a handle takes 0.4 ms to make)
        Blas own;
        rocblas_handle hs = h;
        if (nn > size_t(32) << 20) {
            RSI_BLAS(ctx, rocblas_create_handle(&own.h));
            RSI_BLAS(ctx, rocblas_set_stream(own.h, st));
            hs = own.h;
        }
        RSI_BLAS(ctx, rocsolver_dsyevd(hs, rocblas_evect_original, rocblas_fill_upper, (rocblas_int)naux, dU,
                                       (rocblas_int)naux, dlam, dE, dinfo));
        std::vector<double> lam(naux), w(naux);
        int info = 0;
        RSI_HIP(ctx, hipMemcpyAsync(lam.data(), dlam, naux * sizeof(double), hipMemcpyDeviceToHost, st));
        RSI_HIP(ctx, hipMemcpyAsync(&info, dinfo, sizeof(int), hipMemcpyDeviceToHost, st));
        RSI_HIP(ctx, hipStreamSynchronize(st));
        if (info != 0) return rjk::fail(ctx, RJK_ERR_NOSOLVER, "rocsolver_dsyevd(V) info = " + std::to_string(info));
        kept = 0;
        for (size_t i = 0; i < naux; ++i) {
            if (lam[i] > thr) {
                w[i] = std::pow(lam[i], -0.25);
                ++kept;
            } else {
                w[i] = 0.0;
            }
        }
        RSI_HIP(ctx, hipMemcpyAsync(dw, w.data(), naux * sizeof(double), hipMemcpyHostToDevice, st));
        hipLaunchKernelGGL(k_scale_cols, dim3((unsigned)((naux * naux + 255) / 256)), dim3(256), 0, st, dU, (int)naux,
                           (const double*)dw);
        RSI_HIP(ctx, hipGetLastError());
        const double one_ = 1.0, zero_ = 0.0;
        RSI_BLAS(ctx, rocblas_dgemm(hs, rocblas_operation_none, rocblas_operation_transpose, (rocblas_int)naux,
                                    (rocblas_int)naux, (rocblas_int)naux, &one_, dU, (rocblas_int)naux, dU,
                                    (rocblas_int)naux, &zero_, dVm, (rocblas_int)naux));
        RSI_HIP(ctx, hipStreamSynchronize(st));   // w is a host temporary
    }
    if (nkept) *nkept = kept;
    if (tU.p) (void)hipFree(std::exchange(tU.p, nullptr));
    t_v = now() - t0;

    // the padding of the columns; the slabs' products write the rest
    if (ldb > ctx->npair)
        RSI_HIP(ctx, hipMemset2DAsync(ctx->b64 + ctx->npair, ldb * sizeof(double), 0,
                                      (ldb - ctx->npair) * sizeof(double), naux, st));
    const double one = 1.0, zero = 0.0;
    int status = RJK_OK;
    if (dev3) {
        // device integrals: slab k's kernels and GEMM follow each other on the stream
        if (!dX_ && !temp(tX, xbytes))
            return rjk::fail(ctx, RJK_ERR_NOMEM, "rsi_build_rimatr: device allocation of the integral slab failed");
        double* const dX = (double*)(dX_ ? dX_ : tX.p);
        int r = RJK_OK;
        std::vector<hipEvent_t> ev(2 * (cuts.size() - 1), nullptr);
        for (auto& e : ev) RSI_HIP(ctx, hipEventCreate(&e));
        for (size_t k = 0; k + 1 < cuts.size() && status == RJK_OK; ++k) {
            const size_t q0 = cuts[k] * (cuts[k] + 1) / 2, nq = cuts[k + 1] * (cuts[k + 1] + 1) / 2 - q0;
            (void)hipEventRecord(ev[2 * k], st);
            r = rsi::gpu3c_slab(g.g, k, st, dX, naux);
            (void)hipEventRecord(ev[2 * k + 1], st);
            if (r) {
                status = rjk::fail(ctx, r, "rsi_build_rimatr: three-centre kernel launch failed");
                break;
            }
            if (rocblas_dgemm(h, rocblas_operation_none, rocblas_operation_none, (rocblas_int)nq,
                              (rocblas_int)naux, (rocblas_int)naux, &one, dX, (rocblas_int)nq, dVm, (rocblas_int)naux, &zero, ctx->b64 + q0,
                              (rocblas_int)ldb) != rocblas_status_success)
                status = rjk::fail(ctx, RJK_ERR_HIP, "rocblas_dgemm(B slab) failed");
        }
        const double t1 = now();
        if (hipStreamSynchronize(st) != hipSuccess && status == RJK_OK)
            status = rjk::fail(ctx, RJK_ERR_HIP, "rsi_build_rimatr: device integrals / GEMM failed");
        if (status == RJK_OK)
            for (size_t k = 0; k + 1 < cuts.size(); ++k) {
                float ms = 0.f;
                if (hipEventElapsedTime(&ms, ev[2 * k], ev[2 * k + 1]) == hipSuccess) t_3c += 1e-3 * ms;
            }
        t_gemm = now() - t1;
        for (auto& e : ev) (void)hipEventDestroy(e);
    } else {
        // host integrals (orbital shells beyond d): slab k+1 on the host overlaps slab k's upload and GEMM
        Host hX[2];
        Dev dXh[2];
        hipEvent_t done[2];
        for (int b = 0; b < 2; ++b) {
            RSI_HIP(ctx, hipHostMalloc(&hX[b].p, maxq * naux * sizeof(double), hipHostMallocDefault));
            RSI_HIP(ctx, hipMalloc(&dXh[b].p, maxq * naux * sizeof(double)));
            RSI_HIP(ctx, hipEventCreateWithFlags(&done[b], hipEventDisableTiming));
            RSI_HIP(ctx, hipEventRecord(done[b], st));
        }
        for (size_t k = 0; k + 1 < cuts.size() && status == RJK_OK; ++k) {
            const int b = (int)(k & 1);
            const size_t j0 = cuts[k], j1 = cuts[k + 1];
            const size_t q0 = j0 * (j0 + 1) / 2, nq = j1 * (j1 + 1) / 2 - q0;
            if (hipEventSynchronize(done[b]) != hipSuccess) {   // host buffer b free again
                status = rjk::fail(ctx, RJK_ERR_HIP, "hipEventSynchronize failed");
                break;
            }
            double t1 = now();
            rsi::int3c_slab(*orb, *aux, j0, j1, (double*)hX[b].p);
            t_3c += now() - t1;
            if (hipMemcpyAsync(dXh[b].p, hX[b].p, nq * naux * sizeof(double), hipMemcpyHostToDevice, st) !=
                hipSuccess) {
                status = rjk::fail(ctx, RJK_ERR_HIP, "hipMemcpyAsync(X slab) failed");
                break;
            }
            // B[P][q0+q] = Σ_Q X[Q][q] Vm[Q][P]   (column-major: Bm(nq × naux, ld ldb) = Xm(nq × naux) Vm)
            if (rocblas_dgemm(h, rocblas_operation_none, rocblas_operation_none, (rocblas_int)nq,
                              (rocblas_int)naux, (rocblas_int)naux, &one, (const double*)dXh[b].p, (rocblas_int)nq,
                              dVm, (rocblas_int)naux, &zero, ctx->b64 + q0,
                              (rocblas_int)ldb) != rocblas_status_success) {
                status = rjk::fail(ctx, RJK_ERR_HIP, "rocblas_dgemm(B slab) failed");
                break;
            }
            if (hipEventRecord(done[b], st) != hipSuccess) {
                status = rjk::fail(ctx, RJK_ERR_HIP, "hipEventRecord failed");
                break;
            }
        }
        double t2 = now();
        (void)hipStreamSynchronize(st);
        t_gemm = now() - t2;   // tail of the device work after the last host slab
        for (int b = 0; b < 2; ++b) (void)hipEventDestroy(done[b]);
    }
    if (status != RJK_OK) {
        rsi::set_error(ctx->err);
        return status;
    }
    rc = rjk::finish_b(ctx);
    if (seconds) {
        seconds[0] = t_3c;
        seconds[1] = t_v;
        seconds[2] = t_gemm;
    }
    return rc;
}

extern "C" int rsi_int3c2e_packed_dev(rjk_ctx* ctx, const rsi_basis* orb, const rsi_basis* aux, size_t j0, size_t j1,
                                      double* out_dev) {
    if (!ctx || !orb || !aux || !out_dev) {
        rsi::set_error("rsi_int3c2e_packed_dev: NULL argument");
        return RJK_ERR_ARG;
    }
    if (j0 >= j1 || j1 > orb->nbf || !rsi::on_shell_boundary(*orb, j0) || !rsi::on_shell_boundary(*orb, j1)) {
        rsi::set_error("rsi_int3c2e_packed_dev: [j0, j1) must be a non-empty range on shell boundaries");
        return RJK_ERR_ARG;
    }
    if (!rsi::gpu3c_supported(*orb, *aux)) {
        rsi::set_error("rsi_int3c2e_packed_dev: device kernels cover orbital shells up to d and auxiliary up to g");
        return RJK_ERR_ARG;
    }
    if (hipSetDevice(ctx->device) != hipSuccess) {
        rsi::set_error("rsi_int3c2e_packed_dev: hipSetDevice failed");
        return RJK_ERR_HIP;
    }
    GpuInts g;
    int rc = rsi::gpu3c_init(&g.g, orb, *aux, std::vector<size_t>{j0, j1}, ctx->stream);
    if (!rc) rc = rsi::gpu3c_slab(g.g, 0, ctx->stream, out_dev, aux->nbf);
    if (!rc && hipStreamSynchronize(ctx->stream) != hipSuccess) rc = RJK_ERR_HIP;
    if (rc) rsi::set_error("rsi_int3c2e_packed_dev: device integrals failed (code " + std::to_string(rc) + ")");
    return rc;
}
