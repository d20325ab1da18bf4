// rjk_util.hip — layout and housekeeping kernels: synthetic B fill, packing
// of full B columns (REST ri3fn) into the packed pair layout, padding of
// compact packed columns to the device leading dimension, FP32 copies,
// symmetrisation of D, a plain copy (counter calibration), a finite check and
// the helpers of the density-only K (pivoted Cholesky factor; general D).
#include <algorithm>

#include "rjk_internal.hpp"

namespace rjk {
namespace {

__device__ inline uint64_t mix64(uint64_t z) {
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    return z ^ (z >> 31);
}

__device__ inline void unpair(size_t p, size_t* i, size_t* j) {
    size_t jj = (size_t)((sqrt(8.0 * (double)p + 1.0) - 1.0) * 0.5);
    while (jj * (jj + 1) / 2 > p) --jj;
    while ((jj + 1) * (jj + 2) / 2 <= p) ++jj;
    *j = jj;
    *i = p - jj * (jj + 1) / 2;
}

// b[P][p] = (2u-1)·sqrt(3/naux), u from the hash of the compact flat index;
// padding elements (p >= npair) are zero.
__global__ void k_fill_synth(uint64_t seed, size_t npair, size_t naux, size_t ldb, double* __restrict__ b) {
    size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    size_t total = naux * ldb;
    const double a = sqrt(3.0 / (double)naux);
    for (; t < total; t += (size_t)gridDim.x * blockDim.x) {
        size_t P = t / ldb, p = t % ldb;
        double v = 0.0;
        if (p < npair) {
            uint64_t z = mix64(seed + (P * npair + p + 1) * 0x9E3779B97F4A7C15ULL);
            double u = (double)(z >> 11) * 0x1.0p-53;
            v = (2.0 * u - 1.0) * a;
        }
        b[t] = v;
    }
}

// full column-major B_P (nbf×nbf) -> packed upper (row <= col), padded ld
__global__ void k_pack_ri3fn(const double* __restrict__ b3, size_t nbf, size_t nP, size_t ldb,
                             double* __restrict__ b) {
    size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    size_t total = nP * ldb;
    size_t npair = nbf * (nbf + 1) / 2;
    for (; t < total; t += (size_t)gridDim.x * blockDim.x) {
        size_t P = t / ldb, p = t % ldb;
        double v = 0.0;
        if (p < npair) {
            size_t i, j;
            unpair(p, &i, &j);
            v = b3[P * nbf * nbf + i + j * nbf];
        }
        b[t] = v;
    }
}

__global__ void k_pad_rimatr(const double* __restrict__ src, size_t npair, size_t nP, size_t ldb,
                             double* __restrict__ b) {
    size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    size_t total = nP * ldb;
    for (; t < total; t += (size_t)gridDim.x * blockDim.x) {
        size_t P = t / ldb, p = t % ldb;
        b[t] = (p < npair) ? src[P * npair + p] : 0.0;
    }
}

__global__ void k_to_fp32(const double* __restrict__ b, size_t n, float* __restrict__ out) {
    size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (; t < n; t += (size_t)gridDim.x * blockDim.x) out[t] = (float)b[t];
}

__global__ void k_symmetrize(const double* __restrict__ dm, size_t nbf, double* __restrict__ out) {
    size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nbf * nbf) return;
    size_t i = t % nbf, j = t / nbf;
    out[t] = 0.5 * (dm[i + j * nbf] + dm[j + i * nbf]);
}

__global__ void k_copy16(const uint4* __restrict__ src, uint4* __restrict__ dst, size_t n16) {
    size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (; t < n16; t += (size_t)gridDim.x * blockDim.x) dst[t] = src[t];
}
__global__ void k_copy1(const unsigned char* __restrict__ src, unsigned char* __restrict__ dst, size_t n) {
    size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) dst[t] = src[t];
}

__global__ void k_check_finite(const double* __restrict__ x, size_t n, int* __restrict__ flag) {
    size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    int bad = 0;
    for (; t < n; t += (size_t)gridDim.x * blockDim.x)
        if (!isfinite(x[t])) bad = 1;
    if (bad) *flag = 1;   // benign race: every writer stores 1
}

// Per-block maxima of |D(i,j) − D(j,i)| and |D(i,j)| over a column-major nbf×nbf D:
// out[2·block] and out[2·block+1]; a non-finite entry makes both +inf.
__global__ __launch_bounds__(256) void k_asym_stats(const double* __restrict__ dm, size_t nbf,
                                                    double* __restrict__ out) {
    const size_t n = nbf * nbf;
    double a = 0.0, m = 0.0;
    for (size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (size_t)gridDim.x * blockDim.x) {
        const size_t i = t % nbf, j = t / nbf;
        const double x = dm[t], y = dm[i * nbf + j];
        if (!isfinite(x)) { a = INFINITY; m = INFINITY; continue; }
        a = fmax(a, fabs(x - y));
        m = fmax(m, fabs(x));
    }
    __shared__ double ra[256], rm[256];
    ra[threadIdx.x] = a;
    rm[threadIdx.x] = m;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h) {
            ra[threadIdx.x] = fmax(ra[threadIdx.x], ra[threadIdx.x + h]);
            rm[threadIdx.x] = fmax(rm[threadIdx.x], rm[threadIdx.x + h]);
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        out[2 * blockIdx.x] = ra[0];
        out[2 * blockIdx.x + 1] = rm[0];
    }
}

// Column sets of the general density-only route, row-major [nrow][nk] like C':
// cx[ν][c] = D(ν, c) (column c of the column-major D), cy[ν][c] = δ_νc, both zero
// outside nbf × nbf.
__global__ void k_prep_general(const double* __restrict__ dm, size_t nbf, size_t nk, size_t nrow,
                               double* __restrict__ cx, double* __restrict__ cy) {
    size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nrow * nk) return;
    const size_t c = t % nk, nu = t / nk;
    const bool in = nu < nbf && c < nbf;
    cx[t] = in ? dm[nu + c * nbf] : 0.0;
    cy[t] = (in && nu == c) ? 1.0 : 0.0;
}

// vk[p(i,j)] = scale · G(i, j) for i <= j, G column-major with leading dimension ldg.
__global__ void k_pack_upper(const double* __restrict__ g, size_t nbf, size_t ldg, double scale,
                             double* __restrict__ vk) {
    const size_t npair = nbf * (nbf + 1) / 2;
    size_t p = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= npair) return;
    size_t i, j;
    unpair(p, &i, &j);
    vk[p] = scale * g[i + j * ldg];
}

// Pivoted Cholesky factor of the symmetric part of a column-major nbf × nbf D: L[k][i], D ≈ Σ_k L_k L_kᵀ,
// for the density-only K (an SCF density has rank nocc, and this finds it in nocc steps where an
// eigensolver needs n).  One work-group: a step is a pivot search, one column of D and k products per
// row, too little to spread over CUs; what bounds it is the chain of barriers and L2 latencies, about 4 us a
// step (nbf 192, rank 40: 154 us against 3 ms for the eigenpairs).  The first columns of L stay in
// LDS as well, the products of a row are split over 1024 / nbf threads.
// Stops when the largest remaining diagonal is at most cut·max diag(D); rank -> out[0], or -1 if a
// diagonal falls below −cut·max (D is not positive semidefinite) or kmax columns do not suffice.
// A D that will need more is given up early, so that an attempt in vain stays a small part of the eigenpairs
// that follow it (nbf 256, eigenvalues 0.1 to 1: 128 columns in vain 0.8 ms of 7.9, given up after 8 7.1):
//   a tail: the largest remaining diagonal below kCholTail of the first but above the cut (the last pivots
//     of low-rank densities are 3% of the first or more);
//   the columns so far extrapolated: k of them that take the share f of the trace need k/f in all or more,
//     since later pivots take less (random and molecular densities of rank r: k/f <= r throughout).
constexpr double kCholTail = 1e-4;
constexpr int kCholProbe = 8;        // column after which the rank is extrapolated,
constexpr int kCholProbeMin = 56;    // unless kmax is below this: so few columns cost little
constexpr int kCholThreads = 1024;
constexpr size_t kCholSmall = 256;   // largest nbf of the one-work-group kernel
constexpr int kCholLds = 16384;   // doubles of L kept in LDS
__global__ __launch_bounds__(kCholThreads) void k_pivot_chol(const double* __restrict__ dm, int n, int kmax, double cut,
                                                             double* __restrict__ L, int* __restrict__ out) {
    extern __shared__ double sm[];
    double* ls = sm;                        // [kCholLds]
    double* part = sm + kCholLds;           // [kCholThreads]
    double* lp = part + kCholThreads;       // [kmax] row p of L
    __shared__ double wmax[2][16], wmin[2][16], dg[kCholSmall];   // dg: the remaining diagonal
    __shared__ int widx[2][16];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int klds = kCholLds / n;          // columns of L kept in LDS
    int G = 1;                              // threads that share a row's products: all rows at once (n <= kCholSmall)
    while (2 * G * n <= kCholThreads) G *= 2;
    const int row = tid / G, q = tid % G;
    for (int i = tid; i < n; i += kCholThreads) dg[i] = dm[(size_t)i * n + i];
    __syncthreads();
    double d0 = 0.0, trace0 = 0.0;
    int rank = -1;
    const auto trace = [&]() {
        double s = tid < n ? dg[tid] : 0.0;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
        if (lane == 0) part[wave] = s;
        __syncthreads();
        s = part[lane & 15];
#pragma unroll
        for (int o = 8; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
        __syncthreads();
        return s;
    };
    const bool probe = kmax >= kCholProbeMin;
    if (probe) trace0 = trace();
    for (int k = 0;; ++k) {
        if (probe && k == kCholProbe && k * trace0 > kmax * (trace0 - trace())) break;
        double mx = -INFINITY, mn = INFINITY;
        int at = 0;
        for (int i = tid; i < n; i += kCholThreads) {
            const double d = dg[i];
            if (d > mx) {
                mx = d;
                at = i;
            }
            mn = fmin(mn, d);
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            const double m2 = __shfl_xor(mx, o, 64);
            const int a2 = __shfl_xor(at, o, 64);
            if (m2 > mx || (m2 == mx && a2 < at)) {
                mx = m2;
                at = a2;
            }
            mn = fmin(mn, __shfl_xor(mn, o, 64));
        }
        if (lane == 0) {
            wmax[k & 1][wave] = mx;
            wmin[k & 1][wave] = mn;
            widx[k & 1][wave] = at;
        }
        __syncthreads();
        mx = wmax[k & 1][lane & 15];   // every wave finishes for itself
        mn = wmin[k & 1][lane & 15];
        at = widx[k & 1][lane & 15];
#pragma unroll
        for (int o = 8; o > 0; o >>= 1) {
            const double m2 = __shfl_xor(mx, o, 64);
            const int a2 = __shfl_xor(at, o, 64);
            if (m2 > mx || (m2 == mx && a2 < at)) {
                mx = m2;
                at = a2;
            }
            mn = fmin(mn, __shfl_xor(mn, o, 64));
        }
        const double top = mx, low = mn;
        const int p = at;
        if (k == 0) d0 = top;
        if (low < -cut * d0 || !(top >= 0.0)) break;      // not positive semidefinite (or NaN)
        if (top <= cut * d0) {
            rank = k;
            break;
        }
        if (k == kmax || top < kCholTail * d0) break;
        // D's column is on its way while row p of L is gathered and multiplied
        const double dcol = q == 0 && row < n ? 0.5 * (dm[(size_t)p * n + row] + dm[(size_t)row * n + p]) : 0.0;
        for (int j = tid; j < k; j += kCholThreads) lp[j] = j < klds ? ls[j * n + p] : L[(size_t)j * n + p];
        __syncthreads();
        double v = 0.0;
        if (row < n) {
            const int kl = min(k, klds);
            int j = q;
            for (; j < kl; j += G) v += ls[j * n + row] * lp[j];
            for (; j + 7 * G < k; j += 8 * G) {   // eight loads in flight
                double x[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) x[u] = L[(size_t)(j + u * G) * n + row];
#pragma unroll
                for (int u = 0; u < 8; ++u) v += x[u] * lp[j + u * G];
            }
            for (; j < k; j += G) v += L[(size_t)j * n + row] * lp[j];
        }
        part[tid] = v;
        __syncthreads();
        if (q == 0 && row < n) {
            for (int u = 1; u < G; ++u) v += part[tid + u];
            const double inv = 1.0 / sqrt(top);
            const double l = row == p ? top * inv : (dcol - v) * inv;
            if (k < klds) ls[k * n + row] = l;
            L[(size_t)k * n + row] = l;
            dg[row] = row == p ? 0.0 : dg[row] - l * l;
        }
        __syncthreads();
    }
    if (tid == 0) out[0] = rank;
}

// Step k of the same factor for larger D, one launch a step and 64 rows a work-group: the row of products
// is rank·nbf reads, 26 us a step at nbf 1536 on one CU.  Every work-group finds the pivot in diag[k % 2] by
// itself and writes its rows' diagonals to the other half; out[k % 2] is the state launch k finds: −2 running,
// else the verdict of an earlier launch, which it hands on.
constexpr int kCholRows = 64;
__global__ void k_chol_start(const double* __restrict__ dm, int n, double* __restrict__ diag, int* __restrict__ out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) diag[i] = dm[(size_t)i * n + i];
    if (i == 0) out[0] = -2;
    if (i == 1) out[1] = -2;
}
__global__ __launch_bounds__(256) void k_chol_step(const double* __restrict__ dm, int n, int k, int kmax, double cut,
                                                   double* __restrict__ diag, double* __restrict__ top0,
                                                   double* __restrict__ L, int* __restrict__ out) {
    __shared__ double wmax[4], wmin[4], wsum[4], part[256], lp[kCholMaxRank];
    __shared__ int widx[4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (out[k & 1] != -2) {   // finished in an earlier launch (uniform): hand the verdict on
        if (blockIdx.x == 0 && tid == 0) out[(k + 1) & 1] = out[k & 1];
        return;
    }
    const double* __restrict__ din = diag + (size_t)(k & 1) * n;
    double mx = -INFINITY, mn = INFINITY, sum = 0.0;
    int at = 0;
    for (int i = tid; i < n; i += 256) {
        const double d = din[i];
        sum += d;
        if (d > mx) {
            mx = d;
            at = i;
        }
        mn = fmin(mn, d);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const double m2 = __shfl_xor(mx, o, 64);
        const int a2 = __shfl_xor(at, o, 64);
        if (m2 > mx || (m2 == mx && a2 < at)) {
            mx = m2;
            at = a2;
        }
        mn = fmin(mn, __shfl_xor(mn, o, 64));
        sum += __shfl_xor(sum, o, 64);
    }
    if (lane == 0) {
        wmax[wave] = mx;
        wmin[wave] = mn;
        wsum[wave] = sum;
        widx[wave] = at;
    }
    __syncthreads();
    double top = wmax[0], low = wmin[0];
    int p = widx[0];
    for (int w = 1; w < 4; ++w) {
        if (wmax[w] > top) {
            top = wmax[w];
            p = widx[w];
        }
        low = fmin(low, wmin[w]);
    }
    const double d0 = k == 0 ? top : top0[0];
    const bool bad = low < -cut * d0 || !(top >= 0.0), done = top <= cut * d0;
    sum = (wsum[0] + wsum[1]) + (wsum[2] + wsum[3]);
    const bool over = k == kmax || top < kCholTail * d0 ||
                      (k == kCholProbe && k * top0[1] > kmax * (top0[1] - sum));
    if (blockIdx.x == 0 && tid == 0) {
        if (k == 0) {
            top0[0] = top;
            top0[1] = sum;
        }
        out[(k + 1) & 1] = bad ? -1 : (done ? k : (over ? -1 : -2));   // the next launch's state
    }
    if (bad || done || over) return;   // uniform over the grid
    for (int j = tid; j < k; j += 256) lp[j] = L[(size_t)j * n + p];
    __syncthreads();
    const int i = blockIdx.x * kCholRows + lane;
    double v = 0.0;
    if (i < n) {
        int j = wave;
        for (; j + 28 < k; j += 32) {   // eight loads in flight
            double x[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) x[u] = L[(size_t)(j + 4 * u) * n + i];
#pragma unroll
            for (int u = 0; u < 8; ++u) v += x[u] * lp[j + 4 * u];
        }
        for (; j < k; j += 4) v += L[(size_t)j * n + i] * lp[j];
    }
    part[tid] = v;
    __syncthreads();
    if (wave == 0 && i < n) {
        v = (part[lane] + part[lane + 64]) + (part[lane + 128] + part[lane + 192]);
        const double inv = 1.0 / sqrt(top);
        const double l = i == p ? top * inv : (0.5 * (dm[(size_t)p * n + i] + dm[(size_t)i * n + p]) - v) * inv;
        L[(size_t)k * n + i] = l;
        diag[(size_t)((k + 1) & 1) * n + i] = i == p ? 0.0 : din[i] - l * l;
    }
}

// Per-block maxima of |½(D + Dᵀ) − Σ_{k < rank} L_k L_kᵀ|: whether the factor holds all of D.  32 × 32 blocks.
__global__ __launch_bounds__(256) void k_chol_residual(const double* __restrict__ dm, int n, const double* __restrict__ L,
                                                       const int* __restrict__ rank_dev, double* __restrict__ out) {
    __shared__ double la[32][33], lb[32][33], red[256];
    const int rank = rank_dev[0];
    const int bi = blockIdx.x * 32, bj = blockIdx.y * 32;
    const int x = threadIdx.x & 31, y = threadIdx.x >> 5;   // element (bi + x, bj + y + 8 q)
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
    if (bi <= bj)
        for (int k0 = 0; k0 < rank; k0 += 32) {
            for (int r = y; r < 32; r += 8) {
                const int k = k0 + r;
                la[r][x] = (k < rank && bi + x < n) ? L[(size_t)k * n + bi + x] : 0.0;
                lb[r][x] = (k < rank && bj + x < n) ? L[(size_t)k * n + bj + x] : 0.0;
            }
            __syncthreads();
#pragma unroll 8
            for (int r = 0; r < 32; ++r)
#pragma unroll
                for (int q = 0; q < 4; ++q) acc[q] += la[r][x] * lb[r][y + 8 * q];
            __syncthreads();
        }
    double m = 0.0;
    if (bi <= bj)
        for (int q = 0; q < 4; ++q) {
            const int i = bi + x, j = bj + y + 8 * q;
            if (i < n && j < n) m = max_nan(m, fabs(0.5 * (dm[(size_t)j * n + i] + dm[(size_t)i * n + j]) - acc[q]));
        }
    red[threadIdx.x] = m;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h) red[threadIdx.x] = max_nan(red[threadIdx.x], red[threadIdx.x + h]);
        __syncthreads();
    }
    if (threadIdx.x == 0) out[blockIdx.y * gridDim.x + blockIdx.x] = red[0];
}

// out[0] = max of x[0 .. n)
__global__ __launch_bounds__(256) void k_max(const double* __restrict__ x, int n, double* __restrict__ out) {
    __shared__ double red[256];
    double m = 0.0;
    for (int i = threadIdx.x; i < n; i += 256) m = max_nan(m, x[i]);
    red[threadIdx.x] = m;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h) red[threadIdx.x] = max_nan(red[threadIdx.x], red[threadIdx.x + h]);
        __syncthreads();
    }
    if (threadIdx.x == 0) out[0] = red[0];
}

unsigned grid_for(size_t n) {
    size_t g = (n + 255) / 256;
    if (g > 65536) g = 65536;
    if (g == 0) g = 1;
    return (unsigned)g;
}

}  // namespace

hipError_t launch_fill_synth(hipStream_t st, uint64_t seed, size_t npair, size_t naux, size_t ldb, double* b) {
    hipLaunchKernelGGL(k_fill_synth, dim3(grid_for(naux * ldb)), dim3(256), 0, st, seed, npair, naux, ldb, b);
    return hipGetLastError();
}
hipError_t launch_pack_ri3fn(hipStream_t st, const double* b3, size_t nbf, size_t nP, size_t ldb, double* b) {
    hipLaunchKernelGGL(k_pack_ri3fn, dim3(grid_for(nP * ldb)), dim3(256), 0, st, b3, nbf, nP, ldb, b);
    return hipGetLastError();
}
hipError_t launch_pad_rimatr(hipStream_t st, const double* src, size_t npair, size_t nP, size_t ldb, double* b) {
    hipLaunchKernelGGL(k_pad_rimatr, dim3(grid_for(nP * ldb)), dim3(256), 0, st, src, npair, nP, ldb, b);
    return hipGetLastError();
}
hipError_t launch_to_fp32(hipStream_t st, const double* b, size_t n, float* out) {
    hipLaunchKernelGGL(k_to_fp32, dim3(grid_for(n)), dim3(256), 0, st, b, n, out);
    return hipGetLastError();
}
hipError_t launch_symmetrize(hipStream_t st, const double* dm, size_t nbf, double* out) {
    size_t n = nbf * nbf;
    hipLaunchKernelGGL(k_symmetrize, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, dm, nbf, out);
    return hipGetLastError();
}
hipError_t launch_copy(hipStream_t st, void* dst, const void* src, size_t bytes) {
    size_t n16 = bytes / 16;
    if (n16)
        hipLaunchKernelGGL(k_copy16, dim3(grid_for(n16)), dim3(256), 0, st, (const uint4*)src, (uint4*)dst, n16);
    size_t rem = bytes - n16 * 16;
    if (rem)
        hipLaunchKernelGGL(k_copy1, dim3(1), dim3(256), 0, st, (const unsigned char*)src + n16 * 16,
                           (unsigned char*)dst + n16 * 16, rem);
    return hipGetLastError();
}
size_t pivot_chol_lds(size_t kmax) { return (kCholLds + kCholThreads + kmax) * sizeof(double); }
hipError_t launch_pivot_chol(hipStream_t st, const double* dm, size_t nbf, size_t kmax, double cut, double* diag, double* L,
                             int* rank, double* blockmax, double* residual) {
    const size_t lds = pivot_chol_lds(kmax);
    const unsigned nb = (unsigned)((nbf + 31) / 32);
    if (nbf > kCholSmall) {
        int* state = (int*)(blockmax + (size_t)nb * nb);            // two ints
        double* top0 = blockmax + (size_t)nb * nb + 1;
        hipLaunchKernelGGL(k_chol_start, dim3((unsigned)((nbf + 255) / 256)), dim3(256), 0, st, dm, (int)nbf, diag, state);
        const unsigned g = (unsigned)((nbf + kCholRows - 1) / kCholRows);
        for (size_t k = 0; k <= kmax; ++k)
            hipLaunchKernelGGL(k_chol_step, dim3(g), dim3(256), 0, st, dm, (int)nbf, (int)k, (int)kmax, cut, diag, top0,
                               L, state);
        const hipError_t e0 = hipGetLastError();
        if (e0 != hipSuccess) return e0;
        int* verdict = state + ((kmax + 1) & 1);
        hipLaunchKernelGGL(k_chol_residual, dim3(nb, nb), dim3(256), 0, st, dm, (int)nbf, L, verdict, blockmax);
        hipLaunchKernelGGL(k_max, dim3(1), dim3(256), 0, st, blockmax, (int)(nb * nb), residual);
        hipLaunchKernelGGL(k_copy1, dim3(1), dim3(256), 0, st, (const unsigned char*)verdict, (unsigned char*)rank,
                           sizeof(int));
        return hipGetLastError();
    }
    // more LDS than a launch's default limit
    const hipError_t e =
        hipFuncSetAttribute((const void*)k_pivot_chol, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_pivot_chol, dim3(1), dim3(kCholThreads), lds, st, dm, (int)nbf, (int)kmax, cut, L, rank);
    hipLaunchKernelGGL(k_chol_residual, dim3(nb, nb), dim3(256), 0, st, dm, (int)nbf, L, rank, blockmax);
    hipLaunchKernelGGL(k_max, dim3(1), dim3(256), 0, st, blockmax, (int)(nb * nb), residual);
    return hipGetLastError();
}
unsigned asym_stats_blocks(size_t nbf) {
    size_t g = (nbf * nbf + 255) / 256;
    return (unsigned)std::min<size_t>(std::max<size_t>(g, 1), kAsymBlocks);
}
hipError_t launch_asym_stats(hipStream_t st, const double* dm, size_t nbf, double* out) {
    hipLaunchKernelGGL(k_asym_stats, dim3(asym_stats_blocks(nbf)), dim3(256), 0, st, dm, nbf, out);
    return hipGetLastError();
}
hipError_t launch_prep_general(hipStream_t st, const double* dm, size_t nbf, size_t nk, size_t nrow, double* cx,
                               double* cy) {
    size_t n = nrow * nk;
    hipLaunchKernelGGL(k_prep_general, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, dm, nbf, nk, nrow, cx,
                       cy);
    return hipGetLastError();
}
hipError_t launch_pack_upper(hipStream_t st, const double* g, size_t nbf, size_t ldg, double scale, double* vk) {
    size_t n = nbf * (nbf + 1) / 2;
    hipLaunchKernelGGL(k_pack_upper, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, g, nbf, ldg, scale, vk);
    return hipGetLastError();
}
hipError_t launch_check_finite(hipStream_t st, const double* x, size_t n, int* flag) {
    hipLaunchKernelGGL(k_check_finite, dim3(grid_for(n)), dim3(256), 0, st, x, n, flag);
    return hipGetLastError();
}

}  // namespace rjk
