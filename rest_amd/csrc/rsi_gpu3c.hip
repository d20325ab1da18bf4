// rsi_gpu3c.hip — three-centre integrals (μν|P) and the auxiliary metric (P|Q) on the GPU for the B
// producer.
//
// McMurchie–Davidson (rsi_core.hpp) with the auxiliary side in closed form.  A solid harmonic
// Gaussian is S_lm(∇)/(2g)^l of its s Gaussian, and S_lm(∇) f(R²) = 2^l S_lm(R) f^(l)(R²) (Hobson's
// theorem), so the Hermite integral of a pair with centre P and exponent p against the spherical
// auxiliary function (l, m) of exponent g at C is, with α = p g / (p + g) and R = P − C,
//     (α/g)^l ∂^{tuv} [ S_lm(R) R^{(l)}_{000}(R) ],   R^{(n)}_{000} = (−2α)^{n−l} F_n(α R²):
// the Hermite recursion runs over the pair's order only (at most 4, 35 integrals) from Boys orders
// l .. l + 4, and a Leibniz sum with the derivatives of the polynomial S_lm finishes it.
//   k_pair_e    the pair's spherical Hermite coefficients E[tuv][ab] of every primitive pair, once;
//   k_int3c     one wave per (shell pair, 64 auxiliary functions of one l): the pair's data are wave-
//               uniform (scalar loads, scalar operands of the FMAs), lanes are auxiliary functions,
//               and every array index is a compile-time constant (no scratch memory).
// The earlier kernel, one thread per (pair, auxiliary shell) with Cartesian coefficients on both sides and
// its arrays in scratch memory, took 27.9 ms of a build for one water and 73 for twelve (def2-SVP /
// def2-SVP-JKFIT, 30 classes); these take 0.85 and 3.1, the smallest now bound by 36 launches.  The
// metric of twelve waters, 30 ms on the host, takes 0.3.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <utility>
#include <vector>

#include "rjk_internal.hpp"
#include "rsi_core.hpp"
#include "rsi_gpu3c.hpp"
#include "rsi_internal.hpp"

namespace rsi {
namespace {

__host__ __device__ constexpr int nc_(int l) { return (l + 1) * (l + 2) / 2; }
__host__ __device__ constexpr int rbase(int s) { return s * (s + 1) * (s + 2) / 6; }   // entries with t+u+v < s
__host__ __device__ constexpr int ridx(int t, int u, int v) {
    return rbase(t + u + v) + (u + v) * (u + v + 1) / 2 + v;
}
constexpr int fall(int i, int t) { return t == 0 ? 1 : i * fall(i - 1, t - 1); }
constexpr int binom_(int n, int k) { return k == 0 ? 1 : binom_(n - 1, k - 1) * n / k; }
constexpr int min_(int a, int b) { return a < b ? a : b; }
// exponents of flat index i (the inverse of ridx)
struct Tuv {
    int t, u, v;
};
constexpr Tuv tuv(int i) {
    int s = 0;
    while (rbase(s + 1) <= i) ++s;
    int r = i - rbase(s), w = 0;   // w = u + v
    while ((w + 1) * (w + 2) / 2 <= r) ++w;
    const int v = r - w * (w + 1) / 2;
    return Tuv{s - w, w - v, v};
}
// f(integral_constant<int, 0>) .. f(integral_constant<int, N - 1>): every index a compile-time constant, so
// that no array is indexed at run time (such arrays go to scratch memory)
template <class F, int... I>
__device__ __forceinline__ void each_(F&& f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>()), ...);
}
template <int N, class F>
__device__ __forceinline__ void each(F&& f) {
    each_(f, std::make_integer_sequence<int, N>());
}

// F_l .. F_{l+N}(T): the same grid and expansion as rsi::Boys
template <int l, int N>
__device__ __forceinline__ void boys_range(const double* __restrict__ tab, double T, double* F) {
    if (T < Boys::kTMax) {
        const int i = (int)(T / Boys::kStep + 0.5);
        const double dt = i * Boys::kStep - T;
        const double* __restrict__ row = tab + (size_t)i * Boys::kMTab + l;
        double q[Boys::kOrd + 1], v[N + Boys::kOrd + 1];
        q[0] = 1.0;
#pragma unroll
        for (int k = 1; k <= Boys::kOrd; ++k) q[k] = q[k - 1] * (dt * (1.0 / k));
#pragma unroll
        for (int k = 0; k <= N + Boys::kOrd; ++k) v[k] = row[k];
#pragma unroll
        for (int m = 0; m <= N; ++m) {
            double s = v[m];
#pragma unroll
            for (int k = 1; k <= Boys::kOrd; ++k) s += v[m + k] * q[k];
            F[m] = s;
        }
    } else {
        const double e = exp(-T), h = 0.5 / T;
        double f = 0.5 * sqrt(M_PI / T);
#pragma unroll
        for (int m = 0; m < l + N; ++m) {
            if (m >= l) F[m - l] = f;
            f = ((2 * m + 1) * f - e) * h;
        }
        F[N] = f;
    }
}

// ∂^{tuv} of the function whose order-n bases are base[n] = (−2α)^n F_{l+n}, t+u+v <= L, in place
// (level n overwrites level n + 1 in order of decreasing t+u+v)
template <int L>
__device__ __forceinline__ void hermite_r(const double* base, double X, double Y, double Z, double* r) {
    r[0] = base[L];
    each<L>([&](auto nn) {
        constexpr int n = L - 1 - decltype(nn)::value, top = rbase(L - n + 1);
        each<top - 1>([&](auto ii) {
            constexpr int i = top - 1 - decltype(ii)::value;
            constexpr Tuv q = tuv(i);
            double val;
            if constexpr (q.t > 0) {
                val = X * r[ridx(q.t - 1, q.u, q.v)];
                if constexpr (q.t > 1) val += (q.t - 1) * r[ridx(q.t - 2, q.u, q.v)];
            } else if constexpr (q.u > 0) {
                val = Y * r[ridx(q.t, q.u - 1, q.v)];
                if constexpr (q.u > 1) val += (q.u - 1) * r[ridx(q.t, q.u - 2, q.v)];
            } else {
                val = Z * r[ridx(q.t, q.u, q.v - 1)];
                if constexpr (q.v > 1) val += (q.v - 1) * r[ridx(q.t, q.u, q.v - 2)];
            }
            r[i] = val;
        });
        r[0] = base[n];
    });
}

// 1-D Hermite coefficients of a pair, E[(i (LB+1) + j) (LA+LB+1) + t]
template <int LA, int LB>
__device__ __forceinline__ void hermite_e(double p, double XPA, double XPB, double* E) {
    constexpr int N = LA + LB + 1;
    const double oo2p = 0.5 / p;
    each<(LA + 1) * (LB + 1) * N>([&](auto x) {
        constexpr int e = decltype(x)::value, t = e % N, j = e / N % (LB + 1), i = e / N / (LB + 1);
        if constexpr (i == 0 && j == 0) {
            E[e] = t == 0 ? 1.0 : 0.0;
        } else if constexpr (t <= i + j) {
            constexpr int pi = j == 0 ? i - 1 : i, pj = j == 0 ? j : j - 1, o = (pi * (LB + 1) + pj) * N;
            const double X = j == 0 ? XPA : XPB;
            double v = 0.0;
            if constexpr (t <= pi + pj) v = X * E[o + t];
            if constexpr (t > 0) v += oo2p * E[o + t - 1];
            if constexpr (t + 1 <= pi + pj) v += (t + 1) * E[o + t + 1];
            E[e] = v;
        }
    });
}

constexpr double k2Pi52 = 2.0 * 17.493418327624862;   // 2π^{5/2}

// Primitive pairs of the orbital class (LA >= LB): centre and exponent to pp[k], and for function
// pair ab = ma (2 LB + 1) + mb the spherical coefficients E[tuv][ab], times K·2π^{5/2}/p.
// One thread per (primitive pair, ab).
template <int LA, int LB>
__global__ __launch_bounds__(128) void k_pair_e(const GShell* __restrict__ orb, const double* __restrict__ pexp,
                                                const double* __restrict__ pcoef, const double* __restrict__ tsph,
                                                const GPair* __restrict__ pairs, const GPrim* __restrict__ prims,
                                                int nprims, double* __restrict__ pp, double* __restrict__ E) {
    constexpr int LAB = LA + LB, NT = rbase(LAB + 1), NB = 2 * LB + 1, NAB = (2 * LA + 1) * NB;
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (size_t)nprims * NAB) return;
    const int k = (int)(t / NAB), ab = (int)(t % NAB);
    const GPrim pr = prims[k];
    const GPair& P = pairs[pr.pair];
    const GShell& A = orb[P.a];
    const GShell& B = orb[P.b];
    const double a = pexp[A.p0 + pr.ia], b = pexp[B.p0 + pr.ib], p = a + b, mu = a * b / p;
    const double ABx = A.A[0] - B.A[0], ABy = A.A[1] - B.A[1], ABz = A.A[2] - B.A[2];
    const double K = pcoef[A.p0 + pr.ia] * pcoef[B.p0 + pr.ib] * exp(-mu * (ABx * ABx + ABy * ABy + ABz * ABz));
    const double Px = (a * A.A[0] + b * B.A[0]) / p, Py = (a * A.A[1] + b * B.A[1]) / p,
                 Pz = (a * A.A[2] + b * B.A[2]) / p;
    if (ab == 0) {
        double* o = pp + 4 * (size_t)(P.k0 + pr.k);
        o[0] = p;
        o[1] = Px;
        o[2] = Py;
        o[3] = Pz;
    }
    constexpr int N = LAB + 1, NE = (LA + 1) * (LB + 1) * N;
    double Ex[NE], Ey[NE], Ez[NE];
    hermite_e<LA, LB>(p, Px - A.A[0], Px - B.A[0], Ex);
    hermite_e<LA, LB>(p, Py - A.A[1], Py - B.A[1], Ey);
    hermite_e<LA, LB>(p, Pz - A.A[2], Pz - B.A[2], Ez);
    const double* __restrict__ Ta = tsph + A.t0 + (ab / NB) * nc_(LA);
    const double* __restrict__ Tb = tsph + B.t0 + (ab % NB) * nc_(LB);
    double acc[NT];
    each<NT>([&](auto q) { acc[decltype(q)::value] = 0.0; });
    const double f = K * k2Pi52 / p;
    each<nc_(LA) * nc_(LB)>([&](auto c) {
        constexpr int ca = decltype(c)::value / nc_(LB), cb = decltype(c)::value % nc_(LB);
        constexpr Tuv a3 = tuv(rbase(LA) + ca), b3 = tuv(rbase(LB) + cb);
        const double w = Ta[ca] * Tb[cb] * f;
        each<NT>([&](auto q) {
            constexpr Tuv h = tuv(decltype(q)::value);
            if constexpr (h.t <= a3.t + b3.t && h.u <= a3.u + b3.u && h.v <= a3.v + b3.v)
                acc[decltype(q)::value] += w * Ex[(a3.t * (LB + 1) + b3.t) * N + h.t] *
                                           Ey[(a3.u * (LB + 1) + b3.u) * N + h.u] *
                                           Ez[(a3.v * (LB + 1) + b3.v) * N + h.v];
        });
    });
    double* __restrict__ o = E + P.e0 + (size_t)pr.k * NT * NAB + ab;
    each<NT>([&](auto q) { o[(size_t)decltype(q)::value * NAB] = acc[decltype(q)::value]; });
}

// One auxiliary shell of angular momentum L as the "pair" of the metric: E[m][ijk] of order L alone,
// T / (2a)^L times c·2π^{5/2}/a.  One thread per (primitive, m).
template <int L>
__global__ __launch_bounds__(128) void k_shell_e(const GShell* __restrict__ aux, const double* __restrict__ pexp,
                                                 const double* __restrict__ pcoef, const double* __restrict__ tsph,
                                                 const GPair* __restrict__ pairs, const GPrim* __restrict__ prims,
                                                 int nprims, double* __restrict__ pp, double* __restrict__ E) {
    constexpr int NT = nc_(L), NM = 2 * L + 1;
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (size_t)nprims * NM) return;
    const int k = (int)(t / NM), m = (int)(t % NM);
    const GPrim pr = prims[k];
    const GPair& P = pairs[pr.pair];
    const GShell& D = aux[P.a];
    const double a = pexp[D.p0 + pr.ia];
    if (m == 0) {
        double* o = pp + 4 * (size_t)(P.k0 + pr.k);
        o[0] = a;
        for (int d = 0; d < 3; ++d) o[1 + d] = D.A[d];
    }
    double f = pcoef[D.p0 + pr.ia] * k2Pi52 / a;
    for (int i = 0; i < L; ++i) f *= 0.5 / a;
    double* __restrict__ o = E + P.e0 + (size_t)pr.k * NT * NM + m;
    for (int c = 0; c < NT; ++c) o[(size_t)c * NM] = tsph[D.t0 + m * NT + c] * f;
}

// Hermite order range of a pair: 3c pairs use orders 0 .. LAB, a metric shell its own order alone.
// acc[ab] += E[tuv][ab] · ∂^{tuv}[S_lm R^{(l)}] over the primitive pairs and the auxiliary primitives.
template <int LAB, int LOW, int NAB, int LC>
__device__ __forceinline__ void hermite_sum(const double* __restrict__ pp, const double* __restrict__ E, int nk,
                                            const GShell& C, const double* __restrict__ pexp,
                                            const double* __restrict__ pcoef, const double* tc,
                                            const double* __restrict__ boys, double* acc) {
    constexpr int NT = rbase(LAB + 1) - rbase(LOW), NC = nc_(LC), DS = min_(LAB, LC);
    const double cx = C.A[0], cy = C.A[1], cz = C.A[2];
    const int nprim = C.nprim, p0 = C.p0;
    int most = nprim;   // primitives of the wave's longest shell
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) most = max(most, __shfl_xor(most, o, 64));
    most = __builtin_amdgcn_readfirstlane(most);
    for (int k = 0; k < nk; ++k) {
        const double p = pp[4 * k], X = pp[4 * k + 1] - cx, Y = pp[4 * k + 2] - cy, Z = pp[4 * k + 3] - cz;
        const double* __restrict__ Ek = E + (size_t)k * NT * NAB;
        // derivatives of S_lm at R up to order min(LAB, l)
        double sd[rbase(DS + 1)];
        {
            double mono[rbase(LC + 1)];
            mono[0] = 1.0;
            each<rbase(LC + 1) - 1>([&](auto x) {
                constexpr int i = decltype(x)::value + 1;
                constexpr Tuv q = tuv(i);
                if constexpr (q.t > 0) mono[i] = X * mono[ridx(q.t - 1, q.u, q.v)];
                else if constexpr (q.u > 0) mono[i] = Y * mono[ridx(q.t, q.u - 1, q.v)];
                else mono[i] = Z * mono[ridx(q.t, q.u, q.v - 1)];
            });
            each<rbase(DS + 1)>([&](auto x) {
                constexpr Tuv d = tuv(decltype(x)::value);
                double w = 0.0;
                each<NC>([&](auto c) {
                    constexpr Tuv q = tuv(rbase(LC) + decltype(c)::value);
                    if constexpr (q.t >= d.t && q.u >= d.u && q.v >= d.v) {
                        constexpr double cf = (double)(fall(q.t, d.t) * fall(q.u, d.u) * fall(q.v, d.v));
                        w += (tc[decltype(c)::value] * cf) * mono[ridx(q.t - d.t, q.u - d.u, q.v - d.v)];
                    }
                });
                sd[decltype(x)::value] = w;
            });
        }
        for (int ic = 0; ic < most; ++ic) {
            const bool on = ic < nprim;
            const double g = on ? pexp[p0 + ic] : 1.0;
            const double gi = 1.0 / g, pg = p + g, al = p * g / pg;
            double cf = (on ? pcoef[p0 + ic] : 0.0) * gi / sqrt(pg);
#pragma unroll
            for (int i = 0; i < LC; ++i) cf *= al * gi;
            double F[LAB + 1], r[rbase(LAB + 1)];
            boys_range<LC, LAB>(boys, al * (X * X + Y * Y + Z * Z), F);
            double pw = cf;
#pragma unroll
            for (int n = 0; n <= LAB; ++n) {
                F[n] *= pw;
                pw *= -2.0 * al;
            }
            hermite_r<LAB>(F, X, Y, Z, r);
            each<NT>([&](auto x) {
                constexpr int q = decltype(x)::value;
                constexpr Tuv d = tuv(q + rbase(LOW));
                double h = 0.0;
                each<rbase(DS + 1)>([&](auto y) {
                    constexpr Tuv e = tuv(decltype(y)::value);
                    if constexpr (e.t <= d.t && e.u <= d.u && e.v <= d.v) {
                        constexpr double bn = (double)(binom_(d.t, e.t) * binom_(d.u, e.u) * binom_(d.v, e.v));
                        h += (bn * sd[decltype(y)::value]) * r[ridx(d.t - e.t, d.u - e.u, d.v - e.v)];
                    }
                });
#pragma unroll
                for (int ab = 0; ab < NAB; ++ab) acc[ab] += Ek[q * NAB + ab] * h;
            });
        }
    }
}

// Lane -> auxiliary function f = m·nauxl + shell of class l = LC: neighbouring lanes share m mostly
template <int LC>
struct AuxLane {
    int m;
    bool on;
    const GShell* C;
    double tc[nc_(LC)];
    __device__ AuxLane(const GShell* aux, const int* auxl, int nauxl, const double* tsph, int f) {
        const int nf = nauxl * (2 * LC + 1);
        on = f < nf;
        f = min(f, nf - 1);
        m = f / nauxl;
        C = aux + auxl[f % nauxl];
        const double* T = tsph + C->t0 + m * nc_(LC);
#pragma unroll
        for (int c = 0; c < nc_(LC); ++c) tc[c] = T[c];
    }
};

template <int LA, int LB, int LC>
__global__ __launch_bounds__(256) void k_int3c(const GShell* __restrict__ orb, const GShell* __restrict__ aux,
                                               const double* __restrict__ pexp, const double* __restrict__ pcoef,
                                               const double* __restrict__ tsph, const GPair* __restrict__ pairs,
                                               int npairs, const double* __restrict__ pp, const double* __restrict__ E,
                                               const int* __restrict__ auxl, int nauxl,
                                               const double* __restrict__ boys, size_t q0, size_t nq,
                                               double* __restrict__ X) {
    constexpr int NA = 2 * LA + 1, NB = 2 * LB + 1, NAB = NA * NB;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int w = blockIdx.x * 4 + wave, nfb = (nauxl * (2 * LC + 1) + 63) / 64;
    if (w >= npairs * nfb) return;
    const GPair pr = pairs[w % npairs];   // neighbouring waves: neighbouring pairs of the same functions
    const AuxLane<LC> f(aux, auxl, nauxl, tsph, (w / npairs) * 64 + (threadIdx.x & 63));
    double acc[NAB];
#pragma unroll
    for (int k = 0; k < NAB; ++k) acc[k] = 0.0;
    hermite_sum<LA + LB, 0, NAB, LC>(pp + 4 * (size_t)pr.k0, E + pr.e0, pr.nk, *f.C, pexp, pcoef, f.tc, boys, acc);
    if (!f.on) return;
    const int offa = orb[pr.a].off, offb = orb[pr.b].off;
    double* __restrict__ row = X + (size_t)(f.C->off + f.m) * nq;
#pragma unroll
    for (int ma = 0; ma < NA; ++ma)
#pragma unroll
        for (int mb = 0; mb < NB; ++mb) {
            const size_t i = offa + ma, j = offb + mb;
            if (pr.a == pr.b && i > j) continue;
            const size_t q = (i <= j ? j * (j + 1) / 2 + i : i * (i + 1) / 2 + j) - q0;
            row[q] = acc[ma * NB + mb];
        }
}

// (P|Q) of shell P (class LD, wave-uniform) against functions Q of class LC: V[Q + P·n]
template <int LD, int LC>
__global__ __launch_bounds__(256) void k_int2c(const GShell* __restrict__ aux, const double* __restrict__ pexp,
                                               const double* __restrict__ pcoef, const double* __restrict__ tsph,
                                               const GPair* __restrict__ pairs, int npairs,
                                               const double* __restrict__ pp, const double* __restrict__ E,
                                               const int* __restrict__ auxl, int nauxl,
                                               const double* __restrict__ boys, size_t n, double* __restrict__ V) {
    constexpr int NM = 2 * LD + 1;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int w = blockIdx.x * 4 + wave, nfb = (nauxl * (2 * LC + 1) + 63) / 64;
    if (w >= npairs * nfb) return;
    const GPair pr = pairs[w % npairs];
    const AuxLane<LC> f(aux, auxl, nauxl, tsph, (w / npairs) * 64 + (threadIdx.x & 63));
    double acc[NM];
#pragma unroll
    for (int k = 0; k < NM; ++k) acc[k] = 0.0;
    hermite_sum<LD, LD, NM, LC>(pp + 4 * (size_t)pr.k0, E + pr.e0, pr.nk, *f.C, pexp, pcoef, f.tc, boys, acc);
    if (!f.on) return;
    const int offd = aux[pr.a].off;
#pragma unroll
    for (int m = 0; m < NM; ++m) V[(size_t)(offd + m) * n + f.C->off + f.m] = acc[m];
}

unsigned waves4(size_t waves) { return (unsigned)((waves + 3) / 4); }

template <int LA, int LB>
hipError_t launch_pair_e(hipStream_t st, const Gpu3c& g, const GPrim* prims, int nprims, double* pp, double* E) {
    const size_t n = (size_t)nprims * (2 * LA + 1) * (2 * LB + 1);
    hipLaunchKernelGGL((k_pair_e<LA, LB>), dim3((unsigned)((n + 127) / 128)), dim3(128), 0, st, g.orb, g.pexp, g.pcoef,
                       g.tsph, g.pairs, prims, nprims, pp, E);
    return hipGetLastError();
}

template <int LA, int LB, int LC>
hipError_t launch_class(hipStream_t st, const Gpu3c& g, const GPair* pairs, int npairs, const double* pp,
                        const double* E, size_t q0, size_t nq, double* X) {
    const int na = g.aux_cnt[LC];
    if (!na) return hipSuccess;
    const size_t waves = (size_t)npairs * ((na * (2 * LC + 1) + 63) / 64);
    hipLaunchKernelGGL((k_int3c<LA, LB, LC>), dim3(waves4(waves)), dim3(256), 0, st, g.orb, g.aux, g.pexp, g.pcoef,
                       g.tsph, pairs, npairs, pp, E, g.auxl + g.aux_off[LC], na, g.boys, q0, nq, X);
    return hipGetLastError();
}

template <int LA, int LB>
hipError_t launch_pairs(hipStream_t st, const Gpu3c& g, const GPair* pairs, int npairs, const GPrim* prims, int nprims,
                        double* pp, double* E, size_t q0, size_t nq, double* X) {
    hipError_t e = launch_pair_e<LA, LB>(st, g, prims, nprims, pp, E);
    if (e == hipSuccess) e = launch_class<LA, LB, 0>(st, g, pairs, npairs, pp, E, q0, nq, X);
    if (e == hipSuccess) e = launch_class<LA, LB, 1>(st, g, pairs, npairs, pp, E, q0, nq, X);
    if (e == hipSuccess) e = launch_class<LA, LB, 2>(st, g, pairs, npairs, pp, E, q0, nq, X);
    if (e == hipSuccess) e = launch_class<LA, LB, 3>(st, g, pairs, npairs, pp, E, q0, nq, X);
    if (e == hipSuccess) e = launch_class<LA, LB, 4>(st, g, pairs, npairs, pp, E, q0, nq, X);
    return e;
}

template <int LD, int LC>
hipError_t launch_metric(hipStream_t st, const Gpu3c& g, const GPair* pairs, int npairs, const double* pp,
                         const double* E, size_t n, double* V) {
    const int na = g.aux_cnt[LC];
    if (!na) return hipSuccess;
    const size_t waves = (size_t)npairs * ((na * (2 * LC + 1) + 63) / 64);
    hipLaunchKernelGGL((k_int2c<LD, LC>), dim3(waves4(waves)), dim3(256), 0, st, g.aux, g.pexp, g.pcoef, g.tsph, pairs,
                       npairs, pp, E, g.auxl + g.aux_off[LC], na, g.boys, n, V);
    return hipGetLastError();
}

template <int LD>
hipError_t launch_metrics(hipStream_t st, const Gpu3c& g, const GPair* pairs, int npairs, const GPrim* prims,
                          int nprims, double* pp, double* E, size_t n, double* V) {
    const size_t th = (size_t)nprims * (2 * LD + 1);
    hipLaunchKernelGGL((k_shell_e<LD>), dim3((unsigned)((th + 127) / 128)), dim3(128), 0, st, g.aux, g.pexp, g.pcoef,
                       g.tsph, g.mpairs, prims, nprims, pp, E);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = launch_metric<LD, 0>(st, g, pairs, npairs, pp, E, n, V);
    if (e == hipSuccess) e = launch_metric<LD, 1>(st, g, pairs, npairs, pp, E, n, V);
    if (e == hipSuccess) e = launch_metric<LD, 2>(st, g, pairs, npairs, pp, E, n, V);
    if (e == hipSuccess) e = launch_metric<LD, 3>(st, g, pairs, npairs, pp, E, n, V);
    if (e == hipSuccess) e = launch_metric<LD, 4>(st, g, pairs, npairs, pp, E, n, V);
    return e;
}

}  // namespace

bool gpu3c_aux_supported(const Basis& aux) {
    for (const Shell& s : aux.sh)
        if (s.l > kGpuMaxLAux) return false;
    return true;
}

bool gpu3c_supported(const Basis& orb, const Basis& aux) {
    for (const Shell& s : orb.sh)
        if (s.l > kGpuMaxLOrb) return false;
    for (const Shell& s : aux.sh)
        if (s.l > kGpuMaxLAux) return false;
    return true;
}

int gpu3c_init(Gpu3c* g, const Basis* orb, const Basis& aux, const std::vector<size_t>& cuts, hipStream_t st) {
    std::vector<GShell> go, ga;
    std::vector<double> ex, co, ts;
    auto add = [&](const Shell& s, std::vector<GShell>& out) {
        GShell q{};
        for (int d = 0; d < 3; ++d) q.A[d] = s.A[d];
        q.l = s.l;
        q.nprim = s.nprim;
        q.p0 = (int)ex.size();
        q.t0 = (int)ts.size();
        q.off = s.off;
        ex.insert(ex.end(), s.a.begin(), s.a.end());
        co.insert(co.end(), s.c.begin(), s.c.end());
        ts.insert(ts.end(), s.T.begin(), s.T.end());
        out.push_back(q);
    };
    if (orb)
        for (const Shell& s : orb->sh) add(s, go);
    for (const Shell& s : aux.sh) add(s, ga);
    static const std::vector<double> tab = [] {   // the Boys table, the same for every molecule
        const size_t nrow = (size_t)(Boys::kTMax / Boys::kStep) + 2;
        std::vector<double> t(nrow * Boys::kMTab);
        for (size_t i = 0; i < nrow; ++i) Boys::series(i * Boys::kStep, Boys::kMTab - 1, &t[i * Boys::kMTab]);
        return t;
    }();
    // auxiliary shells grouped by l, and each as a "pair" of the metric
    std::vector<int> flat;
    std::vector<GPair> mp;
    std::vector<GPrim> mprim;
    int mk = 0;
    size_t me = 0;
    for (int l = 0; l <= kGpuMaxLAux; ++l) {
        g->aux_off[l] = (int)flat.size();
        g->mprim_off[l] = (int)mprim.size();
        for (size_t i = 0; i < aux.sh.size(); ++i)
            if (aux.sh[i].l == l) {
                const int np = aux.sh[i].nprim;
                for (int k = 0; k < np; ++k) mprim.push_back(GPrim{(int)mp.size(), k, 0, k});
                mp.push_back(GPair{(int)i, 0, mk, np, me});
                mk += np;
                me += (size_t)np * nc_(l) * (2 * l + 1);
                flat.push_back((int)i);
            }
        g->aux_cnt[l] = (int)flat.size() - g->aux_off[l];
        g->mprim_cnt[l] = (int)mprim.size() - g->mprim_off[l];
    }
    // screened shell pairs per slab and class; A is the shell with the larger l
    g->cuts = cuts;
    const size_t nslab = cuts.empty() ? 0 : cuts.size() - 1;
    g->cls_off.assign(nslab * kGpuClasses, 0);
    g->cls_cnt.assign(nslab * kGpuClasses, 0);
    g->prim_off.assign(nslab * kGpuClasses, 0);
    g->prim_cnt.assign(nslab * kGpuClasses, 0);
    g->dropped.assign(nslab, 0);
    std::vector<GPair> all;
    std::vector<GPrim> prims;
    size_t npp = (size_t)mk, ne = me;
    for (size_t k = 0; k < nslab; ++k) {
        std::vector<std::pair<int, int>> cls[kGpuClasses];
        for (int sb = 0; sb < (int)orb->sh.size(); ++sb) {
            const Shell& B = orb->sh[sb];
            if ((size_t)B.off < cuts[k] || (size_t)B.off >= cuts[k + 1]) continue;
            for (int sa = 0; sa <= sb; ++sa) {
                const Shell& A = orb->sh[sa];
                const int la = std::max(A.l, B.l), lb = std::min(A.l, B.l);
                cls[la * (la + 1) / 2 + lb].push_back(A.l >= B.l ? std::make_pair(sa, sb) : std::make_pair(sb, sa));
            }
        }
        int kp = 0;        // slab-relative primitive pairs and coefficients
        size_t ke = 0;
        for (int la = 0; la <= kGpuMaxLOrb; ++la)
            for (int lb = 0; lb <= la; ++lb) {
                const int c = la * (la + 1) / 2 + lb;
                const size_t per = (size_t)rbase(la + lb + 1) * (2 * la + 1) * (2 * lb + 1);
                g->cls_off[k * kGpuClasses + c] = all.size();
                g->prim_off[k * kGpuClasses + c] = prims.size();
                for (const auto& ab : cls[c]) {
                    const Shell &A = orb->sh[ab.first], &B = orb->sh[ab.second];
                    const double AB2 = (A.A[0] - B.A[0]) * (A.A[0] - B.A[0]) + (A.A[1] - B.A[1]) * (A.A[1] - B.A[1]) +
                                       (A.A[2] - B.A[2]) * (A.A[2] - B.A[2]);
                    int nk = 0;
                    for (int ia = 0; ia < A.nprim; ++ia)
                        for (int ib = 0; ib < B.nprim; ++ib) {
                            const double mu = A.a[ia] * B.a[ib] / (A.a[ia] + B.a[ib]);
                            if (std::fabs(A.c[ia] * B.c[ib]) * std::exp(-mu * AB2) < kPairCut) continue;
                            prims.push_back(GPrim{(int)all.size(), ia, ib, nk++});
                        }
                    if (nk == 0) {   // every primitive pair below the cut-off: the slab's columns stay zero
                        ++g->dropped[k];
                        continue;
                    }
                    all.push_back(GPair{ab.first, ab.second, kp, nk, ke});
                    kp += nk;
                    ke += nk * per;
                }
                g->cls_cnt[k * kGpuClasses + c] = all.size() - g->cls_off[k * kGpuClasses + c];
                g->prim_cnt[k * kGpuClasses + c] = prims.size() - g->prim_off[k * kGpuClasses + c];
            }
        npp = std::max(npp, (size_t)kp);
        ne = std::max(ne, ke);
    }
    // one allocation for all tables: [orb | aux | exp | coef | sph | boys | auxl | pairs | prims | metric | pp | E]
    struct Part {
        void** dst;
        const void* src;
        size_t bytes, off;
    };
    std::vector<Part> parts;
    size_t total = 0;
    auto part = [&](void** dst, const void* src, size_t bytes) {
        parts.push_back(Part{dst, src, bytes, total});
        total += (bytes + 255) / 256 * 256;
    };
    part((void**)&g->orb, go.data(), go.size() * sizeof(GShell));
    part((void**)&g->aux, ga.data(), ga.size() * sizeof(GShell));
    part((void**)&g->pexp, ex.data(), ex.size() * sizeof(double));
    part((void**)&g->pcoef, co.data(), co.size() * sizeof(double));
    part((void**)&g->tsph, ts.data(), ts.size() * sizeof(double));
    part((void**)&g->boys, tab.data(), tab.size() * sizeof(double));
    part((void**)&g->auxl, flat.data(), flat.size() * sizeof(int));
    part((void**)&g->pairs, all.data(), all.size() * sizeof(GPair));
    part((void**)&g->prims, prims.data(), prims.size() * sizeof(GPrim));
    part((void**)&g->mpairs, mp.data(), mp.size() * sizeof(GPair));
    part((void**)&g->mprims, mprim.data(), mprim.size() * sizeof(GPrim));
    const size_t up = total;   // what follows is written on the device
    part((void**)&g->pp, nullptr, 4 * npp * sizeof(double));
    part((void**)&g->E, nullptr, ne * sizeof(double));
    if (hipMalloc(&g->arena, std::max<size_t>(total, 256)) != hipSuccess) {
        (void)hipGetLastError();
        g->arena = nullptr;
        return RJK_ERR_NOMEM;
    }
    std::vector<char> host(up);
    for (const Part& q : parts) {
        *q.dst = (char*)g->arena + q.off;
        if (q.src && q.bytes) std::memcpy(host.data() + q.off, q.src, q.bytes);
    }
    if (up && hipMemcpyAsync(g->arena, host.data(), up, hipMemcpyHostToDevice, st) != hipSuccess) return RJK_ERR_HIP;
    // the host copy dies with this call: finish the upload first
    return hipStreamSynchronize(st) == hipSuccess ? RJK_OK : RJK_ERR_HIP;
}

void gpu3c_free(Gpu3c* g) {
    if (g->arena) (void)hipFree(g->arena);
    *g = Gpu3c();
}

int gpu2c(const Gpu3c& g, hipStream_t st, double* V, size_t naux) {
    for (int l = 0; l <= kGpuMaxLAux; ++l) {
        const int np = g.aux_cnt[l];
        if (!np) continue;
        const GPair* pp = g.mpairs + g.aux_off[l];
        const GPrim* pr = g.mprims + g.mprim_off[l];
        const int nr = g.mprim_cnt[l];
        hipError_t e;
        switch (l) {
            case 0: e = launch_metrics<0>(st, g, pp, np, pr, nr, g.pp, g.E, naux, V); break;
            case 1: e = launch_metrics<1>(st, g, pp, np, pr, nr, g.pp, g.E, naux, V); break;
            case 2: e = launch_metrics<2>(st, g, pp, np, pr, nr, g.pp, g.E, naux, V); break;
            case 3: e = launch_metrics<3>(st, g, pp, np, pr, nr, g.pp, g.E, naux, V); break;
            default: e = launch_metrics<4>(st, g, pp, np, pr, nr, g.pp, g.E, naux, V); break;
        }
        if (e != hipSuccess) return RJK_ERR_HIP;
    }
    return RJK_OK;
}

int gpu3c_slab(const Gpu3c& g, size_t k, hipStream_t st, double* X, size_t naux) {
    const size_t j0 = g.cuts[k], j1 = g.cuts[k + 1];
    const size_t q0 = j0 * (j0 + 1) / 2, nq = j1 * (j1 + 1) / 2 - q0;
    // every column is written by some pair unless a pair was screened out
    if (g.dropped[k] && hipMemsetAsync(X, 0, nq * naux * sizeof(double), st) != hipSuccess) return RJK_ERR_HIP;
    for (int c = 0; c < kGpuClasses; ++c) {
        const size_t e = k * kGpuClasses + c;
        const int np = (int)g.cls_cnt[e], nr = (int)g.prim_cnt[e];
        if (!np) continue;
        const GPair* pp = g.pairs + g.cls_off[e];
        const GPrim* pr = g.prims + g.prim_off[e];
        hipError_t r;
        switch (c) {
            case 0: r = launch_pairs<0, 0>(st, g, pp, np, pr, nr, g.pp, g.E, q0, nq, X); break;
            case 1: r = launch_pairs<1, 0>(st, g, pp, np, pr, nr, g.pp, g.E, q0, nq, X); break;
            case 2: r = launch_pairs<1, 1>(st, g, pp, np, pr, nr, g.pp, g.E, q0, nq, X); break;
            case 3: r = launch_pairs<2, 0>(st, g, pp, np, pr, nr, g.pp, g.E, q0, nq, X); break;
            case 4: r = launch_pairs<2, 1>(st, g, pp, np, pr, nr, g.pp, g.E, q0, nq, X); break;
            default: r = launch_pairs<2, 2>(st, g, pp, np, pr, nr, g.pp, g.E, q0, nq, X); break;
        }
        if (r != hipSuccess) return RJK_ERR_HIP;
    }
    return RJK_OK;
}

}  // namespace rsi
