// rjk_kbf.hip — exchange (K) on the BF16 matrix cores with split operands.
//
// Every operand x is carried as S BF16 planes, x ≈ x_0 + … + x_{S-1} with
// x_0 = bf16(x) and x_k = bf16(x − x_0 − … − x_{k-1}) (round to nearest even),
// and a product uses the plane pairs whose plane indices sum to less than S:
//   S = 2:  a0·b0 + a0·b1 + a1·b0                        (3 MFMAs, ~2^-16 relative)
//   S = 3:  a0·b0 + a0·b1 + a1·b0 + a0·b2 + a1·b1 + a2·b0 (6 MFMAs, ~2^-24 relative)
//   S = 1:  a0·b0                                         (1 MFMA, ~2^-8 relative)
// accumulated in FP32 by v_mfma_f32_16x16x32_bf16.  Lane l supplies
// A[l%16][8(l/16)+i] and B[8(l/16)+i][l%16]; register r of lane l receives
// D[4(l/16)+r][l%16] (probed on gfx950).  Split-K partials join an FP64 sum.
//
// Layouts (BF16 planes as 16 × 32 fragments, rjk_bftile.hpp; padding zero; nbf_pad a multiple of
// 128, nk of 32):
//   B planes  [S][naux] of nbf_pad × nbf_pad   full symmetric squares
//   C' planes [S] of nk × nbf_pad              C'ᵀ: column c of C' as a row
//   M' planes [S][Pc] of nbf_pad × nk          c along the rows of a fragment: both SYRK operands
// Stage 1: M'_P[μ][c] = Σ_ν C'ᵀ[c][ν] B_P[ν][μ]                  (128 or 256 μ × up to 192 c tiles)
// Stage 2: Kpart[split][s][ν][μ] (+)= Σ_{P,c} sign_c M'_P[ν][c] M'_P[μ][c]  (128 × 128 upper tiles)
// Stage 3: the FP64 split reduction of rjk_k.hip.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "rjk_bftile.hpp"
#include "rjk_internal.hpp"

namespace rjk {
namespace {

constexpr int kXcdB = 8;

__device__ inline size_t tri_b(size_t j) { return j * (j + 1) / 2; }

template <int S>
__device__ inline void split_d(double x, __bf16* out) {
    double r = x;
#pragma unroll
    for (int k = 0; k < S; ++k) {
        const __bf16 h = (__bf16)(float)r;
        out[k] = h;
        r -= (double)(float)h;
    }
}

// ---- conversions ---------------------------------------------------------------
// B planes of auxiliary columns [P0, P0 + Pc) from the packed FP64 B (upper triangle,
// element (i<=j) at j(j+1)/2 + i)
template <int S>
__global__ void k_bf_planes_b(const double* __restrict__ b64, size_t ldb, int nbf, int nbf_pad, size_t naux,
                              size_t P0, size_t Pc, __bf16* __restrict__ planes) {
    // A wave a fragment (nbf_pad²/512 of them, a multiple of the block's 4): read along the packed
    // column, lanes on ν left of the diagonal and on μ beyond it, and turned through LDS.
    __shared__ double tile[4][16][bft::KM + 1];
    const size_t sq = (size_t)nbf_pad * nbf_pad, per = sq / bft::FRAG, total = Pc * per;
    const int n32 = nbf_pad / bft::KM, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (size_t t0 = (size_t)blockIdx.x * 4; t0 < total; t0 += (size_t)gridDim.x * 4) {
        const size_t P = (t0 + wave) / per;
        const int f = (int)((t0 + wave) % per), mu0 = f / n32 * 16, nu0 = f % n32 * bft::KM;
        const double* __restrict__ col = b64 + (P0 + P) * ldb;
        const bool left = nu0 < mu0;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int e = i * 64 + lane, r = left ? e / bft::KM : e % 16, c = left ? e % bft::KM : e / 16;
            const int mu = mu0 + r, nu = nu0 + c, lo = mu < nu ? mu : nu, hi = mu < nu ? nu : mu;
            tile[wave][r][c] = hi < nbf ? col[tri_b(hi) + lo] : 0.0;
        }
        __syncthreads();
        bft::u4 v[S];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            double a = tile[wave][lane & 15][(lane >> 4) * 8 + 2 * i], b = tile[wave][lane & 15][(lane >> 4) * 8 + 2 * i + 1];
#pragma unroll
            for (int k = 0; k < S; ++k) {   // as bft::split_pair, with the remainders in FP64
                unsigned w = __builtin_bit_cast(unsigned, bft::bf2{(__bf16)(float)a, (__bf16)(float)b});
                asm("" : "+v"(w));
                v[k][i] = w;
                a -= (double)__builtin_bit_cast(float, w << 16);
                b -= (double)__builtin_bit_cast(float, w & 0xffff0000u);
            }
        }
#pragma unroll
        for (int k = 0; k < S; ++k)
            *(bft::u4*)(planes + ((size_t)k * naux + P0 + P) * sq + (size_t)f * bft::FRAG + lane * 8) = v[k];
        __syncthreads();
    }
}

// C'ᵀ planes and sign masks: column c of spin s is orbital (c − off_s) · sqrt|occ|
template <int S>
__global__ void k_bf_prep_c(const double* __restrict__ eigv, int nbf, int nstate, int nw0, int nw1,
                            const double* __restrict__ occ, int nspin, int off0, int off1, int nk, int nbf_pad,
                            __bf16* __restrict__ ct, unsigned short* __restrict__ smask) {
    const size_t total = (size_t)nk * nbf_pad;
    for (size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x; t < total; t += (size_t)gridDim.x * blockDim.x) {
        const int c = (int)(t / nbf_pad), nu = (int)(t % nbf_pad);
        double v = 0.0, w = 0.0;
        int s = -1, o = 0;
        if (c >= off0 && c < off0 + nw0) {
            s = 0;
            o = c - off0;
        } else if (nspin == 2 && c >= off1 && c < off1 + nw1) {
            s = 1;
            o = c - off1;
        }
        if (s >= 0) {
            w = occ[(size_t)s * nstate + o];
            if (nu < nbf) v = eigv[(size_t)s * nbf * nstate + (size_t)o * nbf + nu] * sqrt(fabs(w));
        }
        __bf16 h[S];
        split_d<S>(v, h);
#pragma unroll
        for (int k = 0; k < S; ++k) ct[(size_t)k * total + bft::frag_elem(c, nu, nbf_pad)] = h[k];
        if (nu == 0) smask[c] = w < 0 ? 0x8000 : 0;
    }
}

// C'ᵀ planes of gathered eigenvectors (density-only route): column col_off + q is
// vecs[:, idx[q]] · sqrt|lam[q]|; the other columns must be zero beforehand.
template <int S>
__global__ void k_bf_prep_c_idx(const double* __restrict__ vecs, int nbf, const int* __restrict__ idx,
                                const double* __restrict__ lam, int ncol, int col_off, int nk, int nbf_pad,
                                __bf16* __restrict__ ct, unsigned short* __restrict__ smask) {
    const size_t total = (size_t)ncol * nbf_pad, plane = (size_t)nk * nbf_pad;
    for (size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x; t < total; t += (size_t)gridDim.x * blockDim.x) {
        const int q = (int)(t / nbf_pad), nu = (int)(t % nbf_pad);
        const double w = lam[q];
        const double v = nu < nbf ? vecs[(size_t)idx[q] * nbf + nu] * sqrt(fabs(w)) : 0.0;
        __bf16 h[S];
        split_d<S>(v, h);
        const size_t e = bft::frag_elem(col_off + q, nu, nbf_pad);
#pragma unroll
        for (int k = 0; k < S; ++k) ct[(size_t)k * plane + e] = h[k];
        if (nu == 0) smask[col_off + q] = w < 0 ? 0x8000 : 0;
    }
}

// SYRK tiles, measured in the K build: two planes 128 × 128 on 2 × 4 waves, 64-deep (nbf 768, 160
// columns: 1.20 ms; 32-deep 1.28, 2 × 2 waves 1.31); three planes the same 32-deep (nbf 900, 190
// columns: 4.5 ms; 2 × 2 waves 5.9, 4 × 2 waves 5.3).  Both run at the rate that a large BF16 matrix
// product reaches on this card, whose clock falls under that load (1.5 GHz in the two-plane SYRK).
template <int S> struct KbfTiles;
template <> struct KbfTiles<2> {
    using Syrk = bft::Cfg<2, 128, 128, 2, 4, 64>;   // X = 128 ν, Y = 128 μ
};
template <> struct KbfTiles<1> {
    using Syrk = bft::Cfg<1, 128, 128, 2, 4, 64>;
};
template <> struct KbfTiles<3> {
    using Syrk = bft::Cfg<3, 128, 128, 2, 4, 32>;
};

// ---- stage 1 -------------------------------------------------------------------
// Y fragments from the B planes
template <int S, int FM>
struct PlaneRows {
    struct Raw { bft::u4 v[S]; };
    const __bf16* base;      // first fragment of the wave's rows, plane 0 (uniform)
    size_t plane, row;       // elements between planes and row fragments
    __device__ __forceinline__ void load(int s, Raw (&r)[FM]) const {
        const int lane = threadIdx.x & 63;
#pragma unroll
        for (int k = 0; k < S; ++k)
#pragma unroll
            for (int j = 0; j < FM; ++j)
                r[j].v[k] = bft::ld16(base + k * plane + j * row + (size_t)s * bft::FRAG + lane * 8);
    }
    __device__ __forceinline__ void frag(const Raw& r, bft::bf8 (&f)[S]) const {
#pragma unroll
        for (int k = 0; k < S; ++k) f[k] = __builtin_bit_cast(bft::bf8, r.v[k]);
    }
};

// 1-D grid, XCD-aware: every tile of auxiliary column P runs on XCD P % 8 and the
// column tiles of one μ tile are consecutive there, so they share B's rows in L2.
template <class H>
__global__ __launch_bounds__(H::NT, 2) void k_bf_khalf(const __bf16* __restrict__ bpl, size_t naux, int nbf,
                                                       int nbf_pad, size_t P0, int Pc, int ntm, int ntc,
                                                       const __bf16* __restrict__ ct, int nk,
                                                       __bf16* __restrict__ mpl) {
    constexpr int S = H::S;
    __shared__ __bf16 lds[H::LDS_ELEMS];
    const int w = blockIdx.x, xcd = w % kXcdB, kq = w / kXcdB, per = ntm * ntc;
    const int Pl = (kq / per) * kXcdB + xcd;
    if (Pl >= Pc) return;   // padding work-groups (uniform exit)
    const int rem = kq % per, mt = rem / ntc, c0 = (rem % ntc) * H::TC;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int mu0 = mt * H::TMU + wave * 16 * H::FM;
    const size_t sq = (size_t)nbf_pad * nbf_pad;
    const PlaneRows<S, H::FM> y{bpl + (P0 + Pl) * sq + (size_t)mu0 * nbf_pad, naux * sq, (size_t)16 * nbf_pad};
    bft::f4 acc[H::FX][H::FM];
    // B_P symmetric; padding rows and columns are zero
    bft::half_tile<H, false>(lds, ct, nk, nbf_pad / bft::KM, c0, (nbf + bft::KM - 1) / bft::KM, mu0 < nbf, y, acc, acc);
    if (mu0 >= nbf_pad) return;
    const size_t mplane = (size_t)Pc * nbf_pad * nk;
    __bf16* __restrict__ mP = mpl + (size_t)Pl * nbf_pad * nk;
#pragma unroll
    for (int i = 0; i < H::FX; ++i) {
        if (c0 + i * 16 >= nk) break;
#pragma unroll
        for (int j = 0; j < H::FM; ++j) bft::store_m<S>(mP, mplane, mu0 + j * 16, c0 + i * 16, nk, lane, acc[i][j]);
    }
}

// ---- stage 2 -------------------------------------------------------------------
// 1-D grid of (nslot rounded up to 8) × nspin × ntile2 work-groups (split s
// on XCD s % 8).  Upper tile pairs (μ tile <= ν tile) of 128 × 128.
template <class C>
__global__ __launch_bounds__(C::NT, 4) void k_bf_ksyrk(const __bf16* __restrict__ mpl, int Pc, int nbf,
                                                    int nbf_pad, int nk, int ntile2, int nspin, int off0, int cnt0,
                                                    int off1, int cnt1,
                                                    const unsigned short* __restrict__ smask, int nslot,
                                                    int p_per_split, int beta, double* __restrict__ kpart,
                                                    size_t slot) {
    __shared__ __bf16 lds[C::LDS_ELEMS];
    const int w = blockIdx.x, xcd = w % kXcdB, kq = w / kXcdB;
    const size_t t = (size_t)(kq % ntile2);
    const int rest = kq / ntile2, spin = rest % nspin, split = (rest / nspin) * kXcdB + xcd;
    const int Pb = split * p_per_split, Pe = min(Pc, Pb + p_per_split);
    if (split >= nslot || (beta && Pb >= Pe)) return;   // uniform exit
    size_t tn = (size_t)((sqrt(8.0 * (double)t + 1.0) - 1.0) * 0.5);
    while (tri_b(tn) > t) --tn;
    while (tri_b(tn + 1) <= t) ++tn;
    const size_t tm = t - tri_b(tn);
    const int mu0 = (int)tm * C::WGY, nu0 = (int)tn * C::WGX;
    const int cb = spin == 0 ? off0 : off1, cnt = spin == 0 ? cnt0 : cnt1;
    const size_t mplane = (size_t)Pc * nbf_pad * nk, mP = (size_t)nbf_pad * nk;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, wx = wave % C::WX, wy = wave / C::WX;
    // outputs of this wave: nothing of them is read beyond nbf or below the diagonal
    const int wnu = nu0 + wx * C::FX * 16, wmu = mu0 + wy * C::FY * 16;
    const bool live = wnu < nbf && wmu < nbf && wmu < wnu + C::FX * 16;
    bft::f4 acc[C::FX][C::FY];
    // D[ν][μ] = Σ_c sign_c M'[ν][c] M'[μ][c]
    const __bf16* __restrict__ base = mpl + (size_t)Pb * mP + (size_t)(cb / bft::KM) * bft::FRAG;
    bft::nt_tile<C>(lds, base + (size_t)nu0 * nk, base + (size_t)mu0 * nk, (size_t)16 * nk, mplane, mP, smask + cb,
                    max(0, Pe - Pb), cnt, live, acc);
    if (!live) return;
    double* __restrict__ kp = kpart + ((size_t)split * nspin + spin) * slot;
#pragma unroll
    for (int i = 0; i < C::FX; ++i)
#pragma unroll
        for (int j = 0; j < C::FY; ++j) {
            const int nb = nu0 + (wx * C::FX + i) * 16 + 4 * (lane >> 4);
            const int mu = mu0 + (wy * C::FY + j) * 16 + (lane & 15);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                double* dst = kp + (size_t)(nb + r) * nbf_pad + mu;
                double v = (double)acc[i][j][r];
                if (beta) v += *dst;
                *dst = v;
            }
        }
}

unsigned gs_blocks(size_t n) { return (unsigned)std::max<size_t>(1, std::min<size_t>((n + 255) / 256, 65536)); }

}  // namespace

int bf_planes(int prec) { return prec == RJK_PREC_BF16X3 ? 3 : (prec == RJK_PREC_BF16X1 ? 1 : 2); }

hipError_t launch_bf_planes_b(hipStream_t st, const double* b64, size_t ldb, size_t nbf, size_t nbf_pad,
                              size_t naux, void* planes) {
    // in slabs of auxiliary columns so each launch's grid-stride loop stays short
    const size_t sq = nbf_pad * nbf_pad, slab = std::max<size_t>(1, (size_t(1) << 28) / sq);
    for (size_t P0 = 0; P0 < naux; P0 += slab) {
        const size_t Pc = std::min(slab, naux - P0);
        hipLaunchKernelGGL(k_bf_planes_b<kBfStoredPlanes>, dim3(gs_blocks(Pc * sq / 8)), dim3(256), 0, st, b64, ldb,
                           (int)nbf, (int)nbf_pad, naux, P0, Pc, (__bf16*)planes);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t launch_bf_prep_c(hipStream_t st, int prec, const double* eigv, size_t nbf, size_t nstate,
                            const size_t* nw, const double* occ, int nspin, const KPlan& kp, void* ct, void* smask) {
    const size_t n = kp.nk * kp.nbf_pad;
    const int nw1 = nspin == 2 ? (int)nw[1] : 0;
    auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3(gs_blocks(n)), dim3(256), 0, st, eigv, (int)nbf, (int)nstate, (int)nw[0], nw1,
                           occ, nspin, (int)kp.col_off[0], (int)kp.col_off[1], (int)kp.nk, (int)kp.nbf_pad,
                           (__bf16*)ct, (unsigned short*)smask);
    };
    switch (bf_planes(prec)) {
        case 3: go(k_bf_prep_c<3>); break;
        case 1: go(k_bf_prep_c<1>); break;
        default: go(k_bf_prep_c<2>); break;
    }
    return hipGetLastError();
}

hipError_t launch_bf_prep_c_idx(hipStream_t st, int prec, const double* vecs, size_t nbf, const int* idx,
                                const double* lam, size_t ncol, size_t col_off, const KPlan& kp, void* ct,
                                void* smask) {
    if (ncol == 0) return hipSuccess;
    const size_t n = ncol * kp.nbf_pad;
    auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3(gs_blocks(n)), dim3(256), 0, st, vecs, (int)nbf, idx, lam, (int)ncol,
                           (int)col_off, (int)kp.nk, (int)kp.nbf_pad, (__bf16*)ct, (unsigned short*)smask);
    };
    switch (bf_planes(prec)) {
        case 3: go(k_bf_prep_c_idx<3>); break;
        case 1: go(k_bf_prep_c_idx<1>); break;
        default: go(k_bf_prep_c_idx<2>); break;
    }
    return hipGetLastError();
}

namespace {

template <class H>
hipError_t bf_khalf_t(hipStream_t st, const void* bpl, size_t naux, size_t nbf, size_t P0, size_t Pc, const KPlan& kp,
                      const void* ct, void* mpl) {
    const int ntm = (int)((kp.nbf_pad + H::TMU - 1) / H::TMU), ntc = (int)((kp.nk + H::TC - 1) / H::TC);
    const size_t nwg = ((Pc + kXcdB - 1) / kXcdB * kXcdB) * (size_t)ntm * ntc;
    hipLaunchKernelGGL(k_bf_khalf<H>, dim3((unsigned)nwg), dim3(H::NT), 0, st, (const __bf16*)bpl, naux, (int)nbf,
                       (int)kp.nbf_pad, P0, (int)Pc, ntm, ntc, (const __bf16*)ct, (int)kp.nk, (__bf16*)mpl);
    return hipGetLastError();
}

// Columns go in tiles of up to 12 fragments, all of one width.  12 against 10 (the columns then in two
// tiles): nbf 768, 192 columns 2.33 against 2.59 ms with two planes, 3.98 against 4.16 with three; 16 is no
// faster (nbf 900, 256 columns: 4.61 against 4.12 ms).  Eight waves share C'ᵀ where their 256 rows are
// no great part of nbf and the tile is wide: nbf 645, 160 columns 2.36 against 2.58 ms with three planes,
// nbf 768 two planes 2.09 against 2.16; four at nbf 300 (0.133 against 0.143 ms) and for 6 fragments
// (nbf 900, three planes: 6.43 against 6.81 ms).
template <int S>
hipError_t bf_khalf_s(hipStream_t st, const void* bpl, size_t naux, size_t nbf, size_t P0, size_t Pc, const KPlan& kp,
                      const void* ct, void* mpl) {
    const size_t f = kp.nk / 16, tiles = (f + 11) / 12, fx = round_up((f + tiles - 1) / tiles, 2);
    auto go = [&](auto fx_) -> hipError_t {
        constexpr int FX = decltype(fx_)::value;
        if constexpr (FX >= 8)
            if (nbf > 512) return bf_khalf_t<bft::HalfCfg<S, FX, 2, 8>>(st, bpl, naux, nbf, P0, Pc, kp, ct, mpl);
        return bf_khalf_t<bft::HalfCfg<S, FX, 2, 4>>(st, bpl, naux, nbf, P0, Pc, kp, ct, mpl);
    };
    switch (fx) {
        case 2: return go(std::integral_constant<int, 2>{});
        case 4: return go(std::integral_constant<int, 4>{});
        case 6: return go(std::integral_constant<int, 6>{});
        case 8: return go(std::integral_constant<int, 8>{});
        case 10: return go(std::integral_constant<int, 10>{});
        default: return go(std::integral_constant<int, 12>{});
    }
}

template <class C>
hipError_t bf_ksyrk_t(hipStream_t st, const void* mpl, size_t nbf, size_t Pc, const KPlan& kp, int nspin, const void* smask,
                      int beta, double* kpart) {
    const size_t nt = kp.nbf_pad / C::WGX, nt2 = nt * (nt + 1) / 2;
    const int pps = (int)((Pc + kp.nsplit - 1) / kp.nsplit);
    const size_t nwg = round_up(kp.nslot, kXcdB) * (size_t)nspin * nt2;
    hipLaunchKernelGGL(k_bf_ksyrk<C>, dim3((unsigned)nwg), dim3(C::NT), 0, st, (const __bf16*)mpl, (int)Pc, (int)nbf,
                       (int)kp.nbf_pad, (int)kp.nk, (int)nt2, nspin, (int)kp.col_off[0], (int)kp.col_cnt[0],
                       (int)kp.col_off[1], (int)kp.col_cnt[1], (const unsigned short*)smask, (int)kp.nslot, pps, beta, kpart,
                       kp.nbf_pad * kp.nbf_pad);
    return hipGetLastError();
}

}  // namespace

// Tile preconditions: nbf_pad a multiple of 128 (SYRK tiles; whole waves of half-transform rows), every
// spin's column count a multiple of 32 (one MFMA deep).
hipError_t launch_bf_khalf(hipStream_t st, int prec, const void* bpl, size_t naux, size_t nbf, size_t P0, size_t Pc,
                           const KPlan& kp, const void* ct, void* mpl) {
    switch (bf_planes(prec)) {
        case 3: return bf_khalf_s<3>(st, bpl, naux, nbf, P0, Pc, kp, ct, mpl);
        case 1: return bf_khalf_s<1>(st, bpl, naux, nbf, P0, Pc, kp, ct, mpl);
        default: return bf_khalf_s<2>(st, bpl, naux, nbf, P0, Pc, kp, ct, mpl);
    }
}

hipError_t launch_bf_ksyrk(hipStream_t st, int prec, const void* mpl, size_t nbf, size_t Pc, const KPlan& kp, int nspin,
                           const void* smask, int beta, double* kpart) {
    switch (bf_planes(prec)) {
        case 3: return bf_ksyrk_t<KbfTiles<3>::Syrk>(st, mpl, nbf, Pc, kp, nspin, smask, beta, kpart);
        case 1: return bf_ksyrk_t<KbfTiles<1>::Syrk>(st, mpl, nbf, Pc, kp, nspin, smask, beta, kpart);
        default: return bf_ksyrk_t<KbfTiles<2>::Syrk>(st, mpl, nbf, Pc, kp, nspin, smask, beta, kpart);
    }
}

}  // namespace rjk
