// rjk_eig.hip — eigenpairs of a symmetric FP64 matrix of at most 1024 rows:
//   1. tridiagonal reduction, up to 192 by one work-group with the matrix in its registers, beyond with
//      one launch a column;
//   2. eigenvalues by Sturm counts, a wave an eigenvalue, 64 points a round;
//   3. eigenvectors of the tridiagonal, a wave a vector, from its twisted factors (Parlett and Dhillon,
//      Linear Algebra Appl. 267, 247 (1997));
//   4. one or two Newton–Schulz steps Z ← Z (3 I − ZᵀZ)/2, which make the vectors of close eigenvalues orthogonal
//      again: a gap g leaves them eps ‖T‖/g from it, and mixing them costs a residual of eps ‖T‖;
//   5. the residuals and ZᵀZ decide whether the pairs are good: equal eigenvalues (a gap below about
//      1e-11 ‖T‖) have no such vectors, and the caller then takes divide and conquer on the same T;
//   6. the vectors transformed back, a wave a vector.
// rocSOLVER's dsyevd spends n² / 2 dependent small launches on the reduction and merges on one
// work-group: n 192 526 us here against 3863, n 64 143 against 1316, n 336 2185 against 7028, n 1024 10.2 ms
// against 22.7, with smaller residuals.
#include <hip/hip_runtime.h>

#include <type_traits>
#include <utility>

#include "rjk_internal.hpp"

namespace rjk {
namespace {

template <class F, int... U>
__device__ __forceinline__ void steps(const F& f, std::integer_sequence<int, U...>) {
    (f(std::integral_constant<int, U>()), ...);
}

template <int CTRL>
__device__ __forceinline__ double dpp(double x) {
    typedef int i2 __attribute__((ext_vector_type(2)));
    i2 w = __builtin_bit_cast(i2, x);
    w[0] = __builtin_amdgcn_update_dpp(0, w[0], CTRL, 0xf, 0xf, true);
    w[1] = __builtin_amdgcn_update_dpp(0, w[1], CTRL, 0xf, 0xf, true);
    return __builtin_bit_cast(double, w);
}
constexpr int kXor1 = 0xB1, kXor2 = 0x4E, kHalfMirror = 0x141, kRor8 = 0x128;   // lanes l^1, l^2, 7−l of 8, l^8

// x: rows of 16 lanes (32 lanes) 1, 3 exchanged for rows 0, 2 of y; x + y then holds x's sums over a pair of
// rows in the even ones and y's in the odd ones
template <int BIT>
__device__ __forceinline__ double pair_sum(double x, double y) {
    typedef unsigned u2 __attribute__((ext_vector_type(2)));
    u2 a = __builtin_bit_cast(u2, x), b = __builtin_bit_cast(u2, y);
#pragma unroll
    for (int w = 0; w < 2; ++w) {
        const auto r = BIT == 16 ? __builtin_amdgcn_permlane16_swap(a[w], b[w], false, false)
                                 : __builtin_amdgcn_permlane32_swap(a[w], b[w], false, false);
        a[w] = r[0];
        b[w] = r[1];
    }
    return __builtin_bit_cast(double, a) + __builtin_bit_cast(double, b);
}

__device__ __forceinline__ double wave_sum(double x) {
    x += dpp<kXor1>(x);
    x += dpp<kXor2>(x);
    x += dpp<kHalfMirror>(x);
    x += dpp<kRor8>(x);
    x = pair_sum<16>(x, x);
    return pair_sum<32>(x, x);
}

template <int BIT>
__device__ __forceinline__ double from_partner(double x) {
    if constexpr (BIT == 8) return dpp<kRor8>(x);
    else if constexpr (BIT == 4) return dpp<kHalfMirror>(x);
    else if constexpr (BIT == 2) return dpp<kXor2>(x);
    else return dpp<kXor1>(x);
}

// Sums of M values over each half wave (32 lanes): a lane ends with the sum of value *at, *at < M or none.
// While a lane has several, it hands half of them to its partner, so that an exchange halves the values.
template <int M, int BIT>
__device__ __forceinline__ double half_wave_sums(const double (&s)[M], int lane, int* at) {
    constexpr int H = (M + 1) / 2;
    const bool up = lane & BIT;
    double t[H];
    if constexpr (M > 1) {
#pragma unroll
        for (int q = 0; q < H; ++q) {
            const double hi = q + H < M ? s[q + H < M ? q + H : 0] : 0.0;
            if constexpr (BIT == 16) t[q] = pair_sum<16>(s[q], hi);
            else t[q] = (up ? hi : s[q]) + from_partner<BIT>(up ? s[q] : hi);
        }
        if (up) *at += H;
    } else if constexpr (BIT == 16) {
        t[0] = pair_sum<16>(s[0], s[0]);
    } else {
        t[0] = s[0] + from_partner<BIT>(s[0]);
    }
    if constexpr (BIT > 1) return half_wave_sums<H, BIT / 2>(t, lane, at);
    else return t[0];
}

__device__ __forceinline__ double recip(double q) {   // 1/q to an ulp or two
    double r = __builtin_amdgcn_rcp(q);
    r = fma(r, fma(-q, r, 1.0), r);
    return fma(r, fma(-q, r, 1.0), r);
}

__device__ __forceinline__ double recip_sqrt(double q) {   // 1/sqrt(q) likewise, q > 0
    double r = __builtin_amdgcn_rsq(q);
    r = fma(0.5 * r, fma(-q * r, r, 1.0), r);
    return fma(0.5 * r, fma(-q * r, r, 1.0), r);
}

// A (upper triangle, column-major) -> T = Qᵀ A Q, Q = H_0 H_1 .., H_k = I − tau_k u_k u_kᵀ with u_k (row k of Hv)
// zero up to k, beyond k + 1 the column itself.  The matrix stays in registers, both halves of it: thread (x, y) of
// TX × 32 holds elements (x + TX r, y + 32 c).  A column then costs its own broadcast through LDS,
// A v as sums over half waves, and the rank-two update: two barriers; every wave forms the norms and
// scalars by itself.  Blocks of 32 columns behind column k drop out of the products.  Bound by the
// chain of a column's sums and barriers and by the waves' instructions: n 192 319 us; before the permlane
// sums and selects instead of branches 428 with TX 16, 498 with 32 (which spills), 528 with 8.
template <int NB, int TX>
__global__ __launch_bounds__(TX * 32) void k_tridiag(const double* __restrict__ A, int n, double* __restrict__ d,
                                                     double* __restrict__ e, double* __restrict__ Hv,
                                                     double* __restrict__ tau_out, int* __restrict__ bad) {
    constexpr int NP = NB * 32, NQ = (NB + 1) / 2, NR = NP / TX;
    __shared__ double xs[2][NQ * 64], ps[NQ * 64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, ty = lane & 31, tx = 2 * wave + (lane >> 5);
    double a[NR][NB];
#pragma unroll
    for (int r = 0; r < NR; ++r)
#pragma unroll
        for (int c = 0; c < NB; ++c) {
            const int i = tx + TX * r, j = ty + 32 * c, lo = min(i, j), hi = max(i, j);
            a[r][c] = hi < n ? A[(size_t)hi * n + lo] : 0.0;
        }
    // the elements have arrived: otherwise the loop waits for memory, and so for its own stores, on every column
    // (n 192: 392 us against 319)
#pragma unroll
    for (int r = 0; r < NR; ++r)
#pragma unroll
        for (int c = 0; c < NB; ++c) asm volatile("" : "+v"(a[r][c]));
    if (tid == 0) bad[0] = 0;
    if (NP < NQ * 64 && tid < 32) {   // entries no row has
        xs[0][NP + tid] = xs[1][NP + tid] = 0.0;
        ps[NP + tid] = 0.0;
    }
    steps(
        [&](auto kc_) {
            constexpr int kc = decltype(kc_)::value, MC = NB - kc, R0 = kc * 32 / TX, MR = NR - R0;
            for (int kk = 0; kk < 32; ++kk) {
                const int k = kc * 32 + kk;
                if (k >= n - 2) break;
                double* const x = xs[kk & 1];
                if (ty == kk)
#pragma unroll
                    for (int r = R0; r < NR; ++r) {
                        const int i = tx + TX * r;
                        x[i] = i > k ? a[r][kc] : 0.0;
                        if (i == k) d[k] = a[r][kc];
                    }
                __syncthreads();
                double xq[NQ], nrm = 0.0;
#pragma unroll
                for (int q = 0; q < NQ; ++q) {
                    xq[q] = lane + 64 * q < R0 * TX ? 0.0 : x[lane + 64 * q];
                    nrm += lane + 64 * q == k + 1 ? 0.0 : xq[q] * xq[q];
                }
                const double alpha = x[k + 1];
                double uc[MC];
#pragma unroll
                for (int c = 0; c < MC; ++c) uc[c] = x[ty + 32 * (kc + c)];
                nrm = wave_sum(nrm);
                // u = column − beta e_{k+1}, tau = 2/uᵀu = 1/(|beta| (|beta| + |alpha|))
                double beta = alpha, tau = 0.0;
                if (nrm > 1e-280) {   // less is no part of any matrix whose products are normal numbers
                    const double s2 = fma(alpha, alpha, nrm), len = s2 * recip_sqrt(s2);
                    beta = alpha >= 0.0 ? -len : len;
                    tau = recip(len * (len + fabs(alpha)));
                }
                const double u1 = alpha - beta;   // u at k + 1
#pragma unroll
                for (int q = 0; q < NQ; ++q) {
                    const int i = lane + 64 * q;
                    xq[q] = i == k + 1 ? u1 : xq[q];
                    if (wave == q && i < n) Hv[(size_t)k * n + i] = xq[q];
                }
                if (tid == 0) {
                    e[k] = beta;
                    tau_out[k] = tau;
                }
                double s[MR];
#pragma unroll
                for (int r = 0; r < MR; ++r) s[r] = 0.0;
#pragma unroll
                for (int c = 0; c < MC; ++c) {
                    uc[c] = ty + 32 * (kc + c) == k + 1 ? u1 : uc[c];
#pragma unroll
                    for (int r = 0; r < MR; ++r) s[r] += a[R0 + r][kc + c] * uc[c];
                }
                int at = 0;
                const double y = half_wave_sums<MR, 16>(s, lane, &at);
                if (at < MR) ps[tx + TX * (R0 + at)] = y;   // lanes that share a value write the same
                __syncthreads();
                // w = tau y − K u, K = tau² yᵀu / 2; what this does to rows and columns up to k is never read
                double dot = 0.0;
#pragma unroll
                for (int q = 0; q < NQ; ++q) dot += lane + 64 * q < R0 * TX ? 0.0 : ps[lane + 64 * q] * xq[q];
                double ur[MR], wr[MR];
#pragma unroll
                for (int r = 0; r < MR; ++r) {
                    const int i = tx + TX * (R0 + r);
                    ur[r] = i == k + 1 ? u1 : x[i];
                    wr[r] = ps[i];
                }
                const double K = 0.5 * tau * tau * wave_sum(dot);
#pragma unroll
                for (int r = 0; r < MR; ++r) wr[r] = tau * wr[r] - K * ur[r];
#pragma unroll
                for (int c = 0; c < MC; ++c) {
                    const double wc = tau * ps[ty + 32 * (kc + c)] - K * uc[c];
#pragma unroll
                    for (int r = 0; r < MR; ++r) a[R0 + r][kc + c] -= ur[r] * wc + wr[r] * uc[c];
                }
            }
        },
        std::make_integer_sequence<int, NB>());
#pragma unroll
    for (int r = 0; r < NR; ++r)
#pragma unroll
        for (int c = 0; c < NB; ++c) {
            const int i = tx + TX * r, j = ty + 32 * c;
            if (i == j && i < n && i >= n - 2) d[i] = a[r][c];
            if (i == n - 1 && j == n - 2) e[j] = a[r][c];
        }
}

// The reduction for n > 192, one launch a column: what a column needs of all rows (the dot product that makes
// w of y = A u, the next column, its norm) every work-group computes from y for itself, and one pass over
// its own rows applies the rank-two update and multiplies by the new u.  A: full square, rows
// contiguous; Y and C: [2][n] by parity of k, y_k and the entries of column k + 1 before update k.
// A launch is 4 to 5 us and the pass over the rows, in L2, hides in it.
constexpr int kStepRows = 2;   // of a wave
__global__ __launch_bounds__(256) void k_step_start(const double* __restrict__ A, int n, double* __restrict__ F,
                                                    double* __restrict__ C, int* __restrict__ bad) {
    const size_t t = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (t == 0) bad[0] = 0;
    if (t >= (size_t)n * n) return;
    const int i = (int)(t / n), j = (int)(t % n);
    const double x = A[(size_t)max(i, j) * n + min(i, j)];
    F[t] = x;
    if (i == 0) C[n + j] = x;
}

template <int NQ>
__global__ __launch_bounds__(256) void k_step(double* __restrict__ F, int n, int k, double* __restrict__ d,
                                              double* __restrict__ e, double* __restrict__ tau_out,
                                              double* __restrict__ Hv, double* __restrict__ Y, double* __restrict__ C) {
    __shared__ double vs[NQ * 64], ws[NQ * 64], us[NQ * 64], red[2][4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int i0 = k + 1 + (blockIdx.x * 4 + wave) * kStepRows, q0 = (k + 1) / 64;
    double a[kStepRows][NQ];
#pragma unroll
    for (int r = 0; r < kStepRows; ++r)
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const int j = lane + 64 * q;
            a[r][q] = q >= q0 && i0 + r < n && j < n ? F[(size_t)(i0 + r) * n + j] : 0.0;
        }
    const double* __restrict__ yk = Y + (size_t)((k + 1) & 1) * n;
    const double* __restrict__ ck = C + (size_t)((k + 1) & 1) * n;
    const double tau0 = k ? tau_out[k - 1] : 0.0;
    constexpr int NT = (NQ * 64 + 255) / 256;
    double y[NT], v[NT], x[NT], dot = 0.0;
#pragma unroll
    for (int m = 0; m < NT; ++m) {
        const int i = tid + 256 * m;
        const bool in = i >= k && i < n;
        y[m] = in && k ? yk[i] : 0.0;
        v[m] = in && k ? Hv[(size_t)(k - 1) * n + i] : 0.0;
        x[m] = in ? ck[i] : 0.0;
        dot += y[m] * v[m];
    }
    dot = wave_sum(dot);
    if (lane == 0) red[0][wave] = dot;
    __syncthreads();
    const double K = 0.5 * tau0 * tau0 * ((red[0][0] + red[0][1]) + (red[0][2] + red[0][3]));
#pragma unroll
    for (int m = 0; m < NT; ++m) {
        const int i = tid + 256 * m;
        if (i < NQ * 64) {
            vs[i] = v[m];
            ws[i] = y[m] = tau0 * y[m] - K * v[m];   // y: w from here on
        }
    }
    __syncthreads();
    const double vk = vs[k], wk = ws[k];
    double nrm = 0.0;
#pragma unroll
    for (int m = 0; m < NT; ++m) {
        const int i = tid + 256 * m;
        x[m] -= v[m] * wk + y[m] * vk;
        if (i < NQ * 64) us[i] = i > k ? x[m] : 0.0;
        if (i > k + 1) nrm += x[m] * x[m];
        if (i == k && blockIdx.x == 0) d[k] = x[m];
    }
    nrm = wave_sum(nrm);
    if (lane == 0) red[1][wave] = nrm;
    __syncthreads();
    nrm = (red[1][0] + red[1][1]) + (red[1][2] + red[1][3]);
    const double alpha = us[k + 1];
    double beta = alpha, tau = 0.0;
    if (nrm > 1e-280) {   // as in k_tridiag
        const double s2 = fma(alpha, alpha, nrm), len = s2 * recip_sqrt(s2);
        beta = alpha >= 0.0 ? -len : len;
        tau = recip(len * (len + fabs(alpha)));
    }
    const double u1 = alpha - beta;
    if (blockIdx.x == 0) {
#pragma unroll
        for (int m = 0; m < NT; ++m) {
            const int i = tid + 256 * m;
            if (i < n) Hv[(size_t)k * n + i] = i == k + 1 ? u1 : us[i];
        }
        if (tid == 0) {
            e[k] = beta;
            tau_out[k] = tau;
        }
    }
    double s[kStepRows];
#pragma unroll
    for (int r = 0; r < kStepRows; ++r) s[r] = 0.0;
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        if (q < q0) continue;
        const int j = lane + 64 * q;
        const double vj = vs[j], wj = ws[j], uj = j == k + 1 ? u1 : us[j];
#pragma unroll
        for (int r = 0; r < kStepRows; ++r) {
            const int i = min(i0 + r, n - 1);
            a[r][q] -= vs[i] * wj + ws[i] * vj;
            s[r] += a[r][q] * uj;
        }
    }
#pragma unroll
    for (int r = 0; r < kStepRows; ++r) {
        const int i = i0 + r;
        const double yi = wave_sum(s[r]);
        if (i >= n) continue;
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const int j = lane + 64 * q;
            if (q >= q0 && j < n) F[(size_t)i * n + j] = a[r][q];
            if (j == k + 1) C[(size_t)(k & 1) * n + i] = a[r][q];
            if (i == n - 1 && j == n - 1 && k == n - 2) d[i] = a[r][q];
        }
        if (lane == 0) Y[(size_t)(k & 1) * n + i] = yi;
    }
}

__device__ __forceinline__ double wave_max(double x) {
    for (int o = 32; o > 0; o >>= 1) x = fmax(x, __shfl_xor(x, o, 64));
    return x;
}

// d, e into LDS; the Gershgorin bound of |T|, the same in every lane
template <int NQ>
__device__ __forceinline__ double load_t(const double* __restrict__ d, const double* __restrict__ e, int n, double* ds,
                                         double* es) {
    const int lane = threadIdx.x & 63;
    double b = 0.0;
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const int i = lane + 64 * q;
        ds[i] = i < n ? d[i] : 0.0;
        es[i] = i < n - 1 ? e[i] : 0.0;
        if (i < n) b = fmax(b, fabs(ds[i]) + fabs(es[i]) + (i > 0 ? fabs(e[i - 1]) : 0.0));
    }
    __syncthreads();
    return wave_max(b);
}
constexpr double kPiv = 1e-18;   // pivots below this share of |T| are moved there: within rounding of T

template <int NQ>
__global__ __launch_bounds__(64) void k_tri_values(const double* __restrict__ d, const double* __restrict__ e, int n,
                                                   double* __restrict__ w) {
    __shared__ double ds[NQ * 64], es[NQ * 64];
    const int k = blockIdx.x, lane = threadIdx.x;
    const double t = load_t<NQ>(d, e, n, ds, es), piv = fmax(kPiv * t, 1e-290);
    double lo = -t - 4e-16 * t, hi = t + 4e-16 * t;
    for (int round = 0; round < 12; ++round) {   // each divides the interval by 65
        if (!(hi - lo > 2e-16 * fmax(fabs(lo), fabs(hi)))) break;
        const double step = (hi - lo) * (1.0 / 65.0), x = lo + step * (lane + 1);
        double q = ds[0] - x;
        int cnt = 0;
        for (int i = 1;; ++i) {
            if (fabs(q) < piv) q = -piv;
            cnt += q < 0.0;
            if (i == n) break;
            double r = __builtin_amdgcn_rcp(q);   // one step: to a few ulps, which perturb e² by as much
            r = fma(r, fma(-q, r, 1.0), r);
            q = ds[i] - x - es[i - 1] * es[i - 1] * r;
        }
        const unsigned long long above = __ballot(cnt > k);   // points with more than k eigenvalues below them
        const int m = above ? __builtin_ctzll(above) : 64;
        const double nlo = m > 0 ? lo + step * m : lo, nhi = m < 64 ? lo + step * (m + 1) : hi;
        lo = nlo;
        hi = nhi;
    }
    if (lane == 0) w[k] = 0.5 * (lo + hi);
}

template <int NQ>
__global__ __launch_bounds__(64) void k_tri_vectors(const double* __restrict__ d, const double* __restrict__ e, int n,
                                                    const double* __restrict__ w, double* __restrict__ Z) {
    __shared__ double ds[NQ * 64], es[NQ * 64], f[2][NQ * 64], z[NQ * 64];
    const int k = blockIdx.x, lane = threadIdx.x;
    const double t = load_t<NQ>(d, e, n, ds, es), piv = fmax(kPiv * t, 1e-290), x = w[k];
    if (lane < 2) {   // the pivots from the top (lane 0) and from the bottom (lane 1)
        double q = 0.0;
        for (int m = 0; m < n; ++m) {
            const int i = lane ? n - 1 - m : m;
            const double g = m ? es[lane ? i : i - 1] : 0.0;
            q = ds[i] - x - (m ? g * g * recip(q) : 0.0);
            if (fabs(q) < piv) q = -piv;
            f[lane][i] = q;
        }
    }
    __syncthreads();
    // twist where |D+ + D− − (d − x)| is least
    double best = INFINITY;
    int r = n;
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const int i = lane + 64 * q;
        if (i < n) {
            const double g = fabs(f[0][i] + f[1][i] - (ds[i] - x));
            if (g < best) {
                best = g;
                r = i;
            }
        }
    }
    for (int o = 32; o > 0; o >>= 1) {
        const double b2 = __shfl_xor(best, o, 64);
        const int r2 = __shfl_xor(r, o, 64);
        if (b2 < best || (b2 == best && r2 < r)) {
            best = b2;
            r = r2;
        }
    }
    if (r >= n) r = 0;   // NaN in T: the check finds it
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NQ; ++q) {   // the ratios of neighbouring components
        const int i = lane + 64 * q;
        if (i < n) z[i] = i < r ? -es[i] * recip(f[0][i]) : (i > r ? -es[i - 1] * recip(f[1][i]) : 1.0);
    }
    __syncthreads();
    if (lane < 2) {
        double p = 1.0;
        for (int i = lane ? r + 1 : r - 1; lane ? i < n : i >= 0; i += lane ? 1 : -1) {
            p *= z[i];
            z[i] = p;
        }
    }
    __syncthreads();
    double s = 0.0;
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const int i = lane + 64 * q;
        if (i < n) s += z[i] * z[i];
    }
    s = 1.0 / sqrt(wave_sum(s));
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const int i = lane + 64 * q;
        if (i < n) Z[(size_t)k * n + i] = z[i] * s;
    }
}

typedef double d4 __attribute__((ext_vector_type(4)));

// T = (3 I − ZᵀZ)/2 (GRAM; part: maxima of |ZᵀZ − I|) or out = Z T, 32 × 32 outputs a work-group, 16 × 16 a
// wave straight from memory: the operands are in L2, and a hundred work-groups leave little to gain from LDS.
// The second step (`first`: the first one's maxima) has nothing to do where those are within kEigOrth: then
// T stays and out = Z.
constexpr double kEigRes = 2e-15, kEigOrth = 1e-8;
__device__ __forceinline__ bool within(const double* __restrict__ x, int n, double bound) {   // by a whole wave
    bool ok = true;
    for (int q = threadIdx.x & 63; q < n; q += 64) ok = ok && x[q] <= bound;
    return __all(ok);
}
template <bool GRAM>
__global__ __launch_bounds__(256) void k_eig_mul(const double* __restrict__ Z, const double* __restrict__ T, int n,
                                                 double* __restrict__ out, double* __restrict__ part,
                                                 const double* __restrict__ first) {
    __shared__ double red[4];
    if (first) {
        if (within(first, (int)(gridDim.x * gridDim.y), kEigOrth)) {   // the same in every wave
            if (GRAM) {
                if (threadIdx.x == 0) part[blockIdx.y * gridDim.x + blockIdx.x] = 0.0;
                return;
            }
            for (int e = threadIdx.x; e < 1024; e += 256) {
                const int i = blockIdx.x * 32 + (e & 31), j = blockIdx.y * 32 + (e >> 5);
                if (i < n && j < n) out[(size_t)j * n + i] = Z[(size_t)j * n + i];
            }
            return;
        }
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l16 = lane & 15, g = lane >> 4;
    const int i0 = blockIdx.x * 32 + (wave & 1) * 16, j0 = blockIdx.y * 32 + (wave >> 1) * 16;
    const int i = min(i0 + l16, n - 1), j = min(j0 + l16, n - 1);
    const double* __restrict__ pa = GRAM ? Z + (size_t)i * n : Z + i;
    const double* __restrict__ pb = (GRAM ? Z : T) + (size_t)j * n;
    d4 acc = {0.0, 0.0, 0.0, 0.0};
    constexpr int U = 24;   // two rounds of loads at n 192
    for (int k0 = 0; k0 < n; k0 += 4 * U) {
        double a[U], b[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = k0 + 4 * u + g, kc = min(k, n - 1);
            a[u] = pa[GRAM ? (size_t)kc : (size_t)kc * n];
            b[u] = pb[kc];
            if (k >= n) a[u] = b[u] = 0.0;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[u], b[u], acc, 0, 0, 0);
    }
    double m = 0.0;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int ii = i0 + g + 4 * r, jj = j0 + l16;
        if (ii < n && jj < n) {
            if (GRAM) {
                const double one = ii == jj ? 1.0 : 0.0, dev = fabs(acc[r] - one);
                m = max_nan(m, dev);
                out[(size_t)jj * n + ii] = 1.5 * one - 0.5 * acc[r];
            } else {
                out[(size_t)jj * n + ii] = acc[r];
            }
        }
    }
    if (!GRAM) return;
    for (int o = 32; o > 0; o >>= 1) m = max_nan(m, __shfl_xor(m, o, 64));
    if (lane == 0) red[wave] = m;
    __syncthreads();
    if (threadIdx.x) return;
    for (int q = 1; q < 4; ++q) m = max_nan(m, red[q]);
    part[blockIdx.y * gridDim.x + blockIdx.x] = m;
}

// bad (zero beforehand) = 1 unless every residual |T z − w z| is within kEigRes of |T| and ZᵀZ was within kEigOrth of one
// before the last step
template <int NQ>
__global__ __launch_bounds__(256) void k_tri_check(const double* __restrict__ d, const double* __restrict__ e, int n,
                                                   const double* __restrict__ w, const double* __restrict__ Z,
                                                   const double* __restrict__ part, int np, int* __restrict__ bad) {
    __shared__ double ds[NQ * 64], es[NQ * 64];
    const int lane = threadIdx.x & 63, k = blockIdx.x * 4 + (threadIdx.x >> 6);
    const double t = load_t<NQ>(d, e, n, ds, es);
    if (k >= n) return;
    const double* __restrict__ z = Z + (size_t)k * n;
    const double x = w[k];
    bool ok = within(part, np, kEigOrth);
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const int i = lane + 64 * q;
        if (i >= n) continue;
        double v = (ds[i] - x) * z[i];
        if (i > 0) v += es[i - 1] * z[i - 1];
        if (i < n - 1) v += es[i] * z[i + 1];
        ok = ok && fabs(v) <= kEigRes * t;
    }
    if (!__all(ok) && lane == 0) bad[0] = 1;
}

// Columns of Z <- H_0 .. H_{n−3} Z, a wave a column: n − 2 dot products of n in registers, four or eight
// reflectors loaded ahead.
template <int NQ>
__global__ __launch_bounds__(64) void k_back(double* __restrict__ Z, int n, const double* __restrict__ Hv,
                                             const double* __restrict__ tau) {
    constexpr int U = NQ > 3 ? 4 : 8;
    const int lane = threadIdx.x;
    double* __restrict__ zc = Z + (size_t)blockIdx.x * n;
    double z[NQ], v[U][NQ], t[U];
#pragma unroll
    for (int q = 0; q < NQ; ++q) z[q] = lane + 64 * q < n ? zc[lane + 64 * q] : 0.0;
    auto load = [&](int u, int k) {
#pragma unroll
        for (int q = 0; q < NQ; ++q) v[u][q] = k >= 0 && lane + 64 * q < n ? Hv[(size_t)k * n + lane + 64 * q] : 0.0;
        t[u] = k >= 0 ? tau[k] : 0.0;
    };
#pragma unroll
    for (int u = 0; u < U; ++u) load(u, n - 3 - u);
    for (int k = n - 3; k >= 0; k -= U) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            double s = 0.0;
#pragma unroll
            for (int q = 0; q < NQ; ++q) s += v[u][q] * z[q];
            s = wave_sum(s) * t[u];
#pragma unroll
            for (int q = 0; q < NQ; ++q) z[q] -= s * v[u][q];
            load(u, k - u - U);
        }
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q)
        if (lane + 64 * q < n) zc[lane + 64 * q] = z[q];
}

}  // namespace

namespace {

// NB: register blocks of the reduction, 0 for a launch a column; NQ: elements a lane of a wave's vector
template <int NB, int NQ>
hipError_t eig_run(hipStream_t st, const double* A, int n, double* w, double* Z, double* ws, int* bad) {
    const size_t n2 = (size_t)n * n;
    double *d = ws, *e = ws + n, *tau = ws + 2 * n, *Hv = ws + 3 * n, *Z1 = Hv + n2, *T = Z1 + n2, *part = T + n2;
    const dim3 tiles((unsigned)((n + 31) / 32), (unsigned)((n + 31) / 32)), waves((unsigned)n), w64(64), w256(256);
    const int np = (int)(tiles.x * tiles.y);
    if constexpr (NB > 0) {
        constexpr int TX = 16;
        hipLaunchKernelGGL((k_tridiag<NB, TX>), dim3(1), dim3(TX * 32), 0, st, A, n, d, e, Hv, tau, bad);
    } else {
        double *Y = T, *C = T + 2 * n;   // the working square in Z1
        hipLaunchKernelGGL(k_step_start, dim3((unsigned)((n2 + 255) / 256)), w256, 0, st, A, n, Z1, C, bad);
        for (int k = 0; k <= n - 2; ++k)
            hipLaunchKernelGGL(k_step<NQ>, dim3((unsigned)((n - 1 - k + 4 * kStepRows - 1) / (4 * kStepRows))), w256, 0, st, Z1,
                               n, k, d, e, tau, Hv, Y, C);
    }
    hipLaunchKernelGGL(k_tri_values<NQ>, waves, w64, 0, st, d, e, n, w);
    hipLaunchKernelGGL(k_tri_vectors<NQ>, waves, w64, 0, st, d, e, n, w, Z);
    const double *none = nullptr;
    hipLaunchKernelGGL(k_eig_mul<true>, tiles, w256, 0, st, Z, none, n, T, part, none);
    hipLaunchKernelGGL(k_eig_mul<false>, tiles, w256, 0, st, Z, T, n, Z1, part, none);
    hipLaunchKernelGGL(k_eig_mul<true>, tiles, w256, 0, st, Z1, none, n, T, part + np, part);
    hipLaunchKernelGGL(k_eig_mul<false>, tiles, w256, 0, st, Z1, T, n, Z, part + np, part);
    hipLaunchKernelGGL(k_tri_check<NQ>, dim3((unsigned)(n + 3) / 4), w256, 0, st, d, e, n, w, Z, part + np, np, bad);
    if (n > 2) hipLaunchKernelGGL(k_back<NQ>, waves, w64, 0, st, Z, n, Hv, tau);
    return hipGetLastError();
}

}  // namespace

size_t eig_ws(size_t n) { return 3 * n + 3 * n * n + 2 * ((n + 31) / 32) * ((n + 31) / 32); }

hipError_t launch_eig(hipStream_t st, const double* A, size_t n, double* w, double* Z, double* ws, int* bad) {
    if (n <= 64) return eig_run<2, 1>(st, A, (int)n, w, Z, ws, bad);
    if (n <= 128) return eig_run<4, 2>(st, A, (int)n, w, Z, ws, bad);
    if (n <= 192) return eig_run<6, 3>(st, A, (int)n, w, Z, ws, bad);
    if (n <= 320) return eig_run<0, 5>(st, A, (int)n, w, Z, ws, bad);
    if (n <= 512) return eig_run<0, 8>(st, A, (int)n, w, Z, ws, bad);
    return eig_run<0, 16>(st, A, (int)n, w, Z, ws, bad);
}

hipError_t launch_eig_back(hipStream_t st, double* Z, size_t n, const double* ws) {
    const double *tau = ws + 2 * n, *Hv = ws + 3 * n;
    if (n <= 2) return hipSuccess;
    auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3((unsigned)n), dim3(64), 0, st, Z, (int)n, Hv, tau);
        return hipGetLastError();
    };
    if (n <= 64) return go(k_back<1>);
    if (n <= 128) return go(k_back<2>);
    if (n <= 192) return go(k_back<3>);
    if (n <= 320) return go(k_back<5>);
    if (n <= 512) return go(k_back<8>);
    return go(k_back<16>);
}

}  // namespace rjk
