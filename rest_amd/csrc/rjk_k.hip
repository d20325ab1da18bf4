// rjk_k.hip — exchange (K) build on packed B, occupied-orbital route.
//
//   K_s = scale · upper( Σ_P M_P diag(occ_s) M_Pᵀ ),  M_P = B_P C_s
//
// which is vk_upper_with_ri_v_sync (src/scf_io/mod.rs:2758-2834) evaluated on
// the packed B of vk_upper_with_rimatr_use_dm_only_sync (:2703-2756).
//
// Columns: the occupied columns of all spins are concatenated (one B stream
// serves both spins); column c of spin s holds C[:,c]·sqrt|occ_c| and a sign
// sign_c = sgn(occ_c), so K = Σ_{P,c} sign_c M'_{P,c} M'_{P,c}ᵀ also for the
// signed weights of the density-only route (D = U Λ Uᵀ).
//
// Stage 1 (K-half): M'[P][c][μ] = Σ_ν B_P[μ,ν] C'[ν][c] — a batched FP64-MFMA
//   GEMM.  The A tile is read straight from the packed column and mirrored
//   through the triangle while it is staged into LDS.
// Stage 2 (K-SYRK): Kpart[split][s][ν][μ] (+)= Σ_{P,c} M'[P][c][μ] sign_c M'[P][c][ν]
//   over upper tile pairs (μ-tile <= ν-tile), split-K over P so that the
//   small nbf×nbf output still fills 256 CUs; deterministic (no atomics).
// Stage 3 (K-reduce): vk_s[p(i,j)] = scale · Σ_slot Kpart[slot][s][j][i].
//
// MFMA: v_mfma_f64_16x16x4f64.  Lane l supplies A[l%16][l/16] and
// B[l/16][l%16]; register r of lane l receives D[l/16 + 4r][l%16] (probed on
// gfx950).  Both kernels put the memory-contiguous index (μ) on the D column
// so that 16 consecutive lanes store 128 contiguous bytes.
#include "rjk_ktiles.hpp"

namespace rjk {
namespace {

using namespace kt;

// ---------------------------------------------------------------------------
// Stage 1 kernel: 1-D grid, XCD-aware — every work-group of auxiliary column P
// runs on XCD P % 8, so the μ-tiles × column tiles of one packed column
// share it in that XCD's L2.
// ---------------------------------------------------------------------------
template <typename T, int FM, int FN>
__global__ __launch_bounds__(kBlock, 3) void k_khalf(const T* __restrict__ b, size_t ldb, int nbf, size_t P0, int Pc,
                                                  int ntm, int ntc, const T* __restrict__ cocc, int nk, int ldm,
                                                  T* __restrict__ m) {
    constexpr int TM = 64 * FM, TN = 16 * FN;
    // XCD-aware decode of the linear work-group id
    const int w = blockIdx.x, xcd = w % kXcd, kq = w / kXcd, per = ntm * ntc;
    const int Pl = (kq / per) * kXcd + xcd;
    if (Pl >= Pc) return;                    // padding work-groups (uniform exit)
    const int rem = kq % per, mt = rem / ntc, ct = rem % ntc;
    khalf_tile<T, FM, FN>(b + (P0 + Pl) * ldb, nbf, mt * TM, ct * TN, cocc, nk, ldm, m + (size_t)Pl * nk * ldm,
                          rotation(kq));
}

// ---------------------------------------------------------------------------
// Stage 2 kernel: 1-D grid of (nslot rounded up to 8) × nspin × ntile(ntile+1)/2
// work-groups; split s runs entirely on XCD s % 8, so the M' slab of a split is
// streamed into one L2 and shared by all tiles there.
// ---------------------------------------------------------------------------
template <typename T, int F>
__global__ __launch_bounds__(kBlock) void k_ksyrk(const T* __restrict__ m, int ldm, int nk, int nbf, int Pc,
                                                  int ntile2, int nspin, SyrkCols cols, const T* __restrict__ sign,
                                                  int nslot, int p_per_split, int beta, double* __restrict__ kpart,
                                                  size_t slot) {
    constexpr int Tt = 32 * F;
    // XCD-aware decode: w -> (split on XCD w%8, spin, tile)
    const int w = blockIdx.x, xcd = w % kXcd, kq = w / kXcd;
    const size_t t = (size_t)(kq % ntile2);
    const int rest = kq / ntile2, spin = rest % nspin, split = (rest / nspin) * kXcd + xcd;
    const int Pb = split * p_per_split, Pe = min(Pc, Pb + p_per_split);
    if (split >= nslot || (beta && Pb >= Pe)) return;   // uniform exit
    size_t tm, tn;
    upper_tile(t, &tm, &tn);
    ksyrk_tile<T, F>(m, ldm, nk, nbf, (int)tm * Tt, (int)tn * Tt, cols.off[spin], cols.cnt[spin] / TK, Pb, Pe, sign,
                      beta, kpart + ((size_t)split * nspin + spin) * slot, rotation(kq));
}

// vk = scale · Σ_slot Kpart.  A work-group sums 32 pairs with 8 threads each (slots g, g + 8, ...),
// so that the chain of dependent additions is an eighth of the slot count and the loads of a
// thread overlap: one thread per pair took 280 us for 1024 slots of 24 × 24, this takes 5.
constexpr int kRedPairs = 32, kRedGroups = 8;
__global__ __launch_bounds__(kRedPairs* kRedGroups) void k_kreduce(const double* __restrict__ kpart, int nslot,
                                                                   int nspin, size_t slot, int ldm, size_t npair,
                                                                   double scale, double* __restrict__ vk) {
    __shared__ double sh[kRedGroups][kRedPairs];
    const int x = threadIdx.x % kRedPairs, g = threadIdx.x / kRedPairs;
    const size_t p = (size_t)blockIdx.x * kRedPairs + x;
    const int s = blockIdx.y;
    double acc = 0;
    if (p < npair) {
        size_t i, j;
        upper_tile(p, &i, &j);   // p = tri(j) + i
        const double* __restrict__ src = kpart + (size_t)s * slot + j * ldm + i;
        const size_t step = (size_t)nspin * slot;
        int q = g;
        for (; q + 3 * kRedGroups < nslot; q += 4 * kRedGroups) {
            double v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = src[(size_t)(q + u * kRedGroups) * step];
            acc += (v[0] + v[1]) + (v[2] + v[3]);
        }
        for (; q < nslot; q += kRedGroups) acc += src[(size_t)q * step];
    }
    sh[g][x] = acc;
    __syncthreads();
    if (g == 0 && p < npair) {
        double t = 0;
#pragma unroll
        for (int u = 0; u < kRedGroups; ++u) t += sh[u][x];
        vk[(size_t)s * npair + p] = t * scale;
    }
}

// C'[ν][c] and sign[c] from the orbitals: column c of spin s is orbital
// (c - off_s) scaled by sqrt|occ|; padding columns and rows are zero.
template <typename T>
__global__ void k_prep_cocc(const double* __restrict__ eigv, int nbf, int nstate, int nw0, int nw1,
                            const double* __restrict__ occ, int nspin, int off0, int off1, int nk, int nrow,
                            T* __restrict__ cocc, T* __restrict__ sign) {
    size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (size_t)nrow * nk) return;
    int c = (int)(t % nk), nu = (int)(t / nk);
    double v = 0.0, sg = 0.0;
    int s = -1, o = 0;
    if (c >= off0 && c < off0 + nw0) { s = 0; o = c - off0; }
    else if (nspin == 2 && c >= off1 && c < off1 + nw1) { s = 1; o = c - off1; }
    if (s >= 0) {
        double w = occ[(size_t)s * nstate + o];
        sg = (w > 0) ? 1.0 : ((w < 0) ? -1.0 : 0.0);
        if (nu < nbf) v = eigv[(size_t)s * nbf * nstate + (size_t)o * nbf + nu] * sqrt(fabs(w));
    }
    cocc[t] = (T)v;
    if (nu == 0) sign[c] = (T)sg;
}

// Columns gathered by index (density-only route): column col_off+q is
// vecs[:, idx[q]] · sqrt|lam[q]|.
template <typename T>
__global__ void k_prep_cocc_idx(const double* __restrict__ vecs, int nbf, const int* __restrict__ idx,
                                const double* __restrict__ lam, int ncol, int col_off, int nk, int nrow,
                                T* __restrict__ cocc, T* __restrict__ sign) {
    size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (size_t)nrow * ncol) return;
    int q = (int)(t % ncol), nu = (int)(t / ncol);
    double w = lam[q];
    double v = (nu < nbf) ? vecs[(size_t)idx[q] * nbf + nu] * sqrt(fabs(w)) : 0.0;
    cocc[(size_t)nu * nk + col_off + q] = (T)v;
    if (nu == 0) sign[col_off + q] = (T)((w > 0) ? 1.0 : ((w < 0) ? -1.0 : 0.0));
}

// C'[ν][c] from columns that are weights already (rows of f, spin s at f + s·fs): the Cholesky factor
// of a density; padding columns and rows are zero
__global__ void k_prep_factor(const double* __restrict__ f, int nbf, size_t fs, int n0, int n1, int off1, int nk,
                              int nrow, double* __restrict__ cocc, double* __restrict__ sign) {
    size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (size_t)nrow * nk) return;
    const int c = (int)(t % nk), nu = (int)(t / nk);
    const bool in0 = c < n0, in1 = c >= off1 && c < off1 + n1;
    const double* src = in0 ? f + (size_t)c * nbf : f + fs + (size_t)(c - off1) * nbf;
    cocc[t] = (in0 || in1) && nu < nbf ? src[nu] : 0.0;
    if (nu == 0) sign[c] = in0 || in1 ? 1.0 : 0.0;
}

template <typename T, int FM, int FN>
hipError_t khalf_go(hipStream_t st, const T* b, size_t ldb, size_t nbf, size_t P0, size_t Pc, const KPlan& kp,
                    const T* cocc, T* m) {
    constexpr int TM = 64 * FM, TN = 16 * FN;
    const int ntm = (int)((nbf + TM - 1) / TM), ntc = (int)(kp.nk / TN);
    const size_t nwg = round_up(Pc, kXcd) * (size_t)ntm * ntc;
    hipLaunchKernelGGL((k_khalf<T, FM, FN>), dim3((unsigned)nwg), dim3(kBlock), 0, st, b, ldb, (int)nbf, P0,
                       (int)Pc, ntm, ntc, cocc, (int)kp.nk, (int)kp.nbf_pad, m);
    return hipGetLastError();
}

// 64-row tiles where nbf fits one, else 128-row ones
template <typename T, int FN>
hipError_t khalf_fm(hipStream_t st, const T* b, size_t ldb, size_t nbf, size_t P0, size_t Pc, const KPlan& kp,
                    const T* cocc, T* m) {
    if (nbf <= 64) return khalf_go<T, 1, FN>(st, b, ldb, nbf, P0, Pc, kp, cocc, m);
    return khalf_go<T, 2, FN>(st, b, ldb, nbf, P0, Pc, kp, cocc, m);
}

template <typename T>
hipError_t khalf_t(hipStream_t st, const T* b, size_t ldb, size_t nbf, size_t P0, size_t Pc, const KPlan& kp,
                   const T* cocc, T* m) {
    switch (kp.fn) {
        case 1: return khalf_fm<T, 1>(st, b, ldb, nbf, P0, Pc, kp, cocc, m);
        case 2: return khalf_fm<T, 2>(st, b, ldb, nbf, P0, Pc, kp, cocc, m);
        case 3: return khalf_fm<T, 3>(st, b, ldb, nbf, P0, Pc, kp, cocc, m);
        case 4: return khalf_fm<T, 4>(st, b, ldb, nbf, P0, Pc, kp, cocc, m);
        case 5: return khalf_fm<T, 5>(st, b, ldb, nbf, P0, Pc, kp, cocc, m);
        case 6:
            if constexpr (sizeof(T) == 4) return khalf_fm<T, 6>(st, b, ldb, nbf, P0, Pc, kp, cocc, m);
            break;
        case 8:
            if constexpr (sizeof(T) == 4) return khalf_fm<T, 8>(st, b, ldb, nbf, P0, Pc, kp, cocc, m);
            break;
    }
    return hipErrorInvalidValue;
}

template <typename T, int F>
hipError_t ksyrk_go(hipStream_t st, const T* m, size_t nbf, size_t Pc, const KPlan& kp, int nspin, const T* sign,
                    int beta, double* kpart) {
    const size_t nt = kp.nbf_pad / (32 * F), nt2 = nt * (nt + 1) / 2;
    SyrkCols cols;
    cols.off[0] = (int)kp.col_off[0];
    cols.cnt[0] = (int)kp.col_cnt[0];
    cols.off[1] = (int)kp.col_off[1];
    cols.cnt[1] = (int)kp.col_cnt[1];
    const int pps = (int)((Pc + kp.nsplit - 1) / kp.nsplit);
    const size_t nwg = round_up(kp.nslot, kXcd) * (size_t)nspin * nt2;
    hipLaunchKernelGGL((k_ksyrk<T, F>), dim3((unsigned)nwg), dim3(kBlock), 0, st, m, (int)kp.nbf_pad, (int)kp.nk,
                       (int)nbf, (int)Pc, (int)nt2, nspin, cols, sign, (int)kp.nslot, pps, beta, kpart,
                       kp.nbf_pad * kp.nbf_pad);
    return hipGetLastError();
}

template <typename T>
hipError_t ksyrk_t(hipStream_t st, const T* m, size_t nbf, size_t Pc, const KPlan& kp, int nspin, const T* sign,
                   int beta, double* kpart) {
    if constexpr (sizeof(T) == 8)
        if (kp.tile == 128) return ksyrk_go<T, 4>(st, m, nbf, Pc, kp, nspin, sign, beta, kpart);
    return ksyrk_go<T, 2>(st, m, nbf, Pc, kp, nspin, sign, beta, kpart);
}

}  // namespace

size_t k_elem_size(int prec) {
    if (is_bf16(prec)) return 2 * (size_t)bf_planes(prec);
    return prec == RJK_PREC_FP64 ? sizeof(double) : sizeof(float);
}

hipError_t launch_prep_cocc(hipStream_t st, int prec, const double* eigv, size_t nbf, size_t nstate,
                            const size_t* nw, const double* occ, int nspin, const KPlan& kp, void* cocc,
                            void* sign) {
    size_t n = kp.nbf_pad * kp.nk;
    dim3 g((unsigned)((n + 255) / 256));
    if (prec == RJK_PREC_FP64)
        hipLaunchKernelGGL(k_prep_cocc<double>, g, dim3(256), 0, st, eigv, (int)nbf, (int)nstate, (int)nw[0],
                           nspin == 2 ? (int)nw[1] : 0, occ, nspin, (int)kp.col_off[0], (int)kp.col_off[1],
                           (int)kp.nk, (int)kp.nbf_pad, (double*)cocc, (double*)sign);
    else
        hipLaunchKernelGGL(k_prep_cocc<float>, g, dim3(256), 0, st, eigv, (int)nbf, (int)nstate, (int)nw[0],
                           nspin == 2 ? (int)nw[1] : 0, occ, nspin, (int)kp.col_off[0], (int)kp.col_off[1],
                           (int)kp.nk, (int)kp.nbf_pad, (float*)cocc, (float*)sign);
    return hipGetLastError();
}

hipError_t launch_prep_cocc_idx(hipStream_t st, int prec, const double* vecs, size_t nbf, const int* idx,
                                const double* lam, size_t ncol, size_t col_off, const KPlan& kp, void* cocc,
                                void* sign) {
    if (ncol == 0) return hipSuccess;
    size_t n = kp.nbf_pad * ncol;
    dim3 g((unsigned)((n + 255) / 256));
    if (prec == RJK_PREC_FP64)
        hipLaunchKernelGGL(k_prep_cocc_idx<double>, g, dim3(256), 0, st, vecs, (int)nbf, idx, lam, (int)ncol,
                           (int)col_off, (int)kp.nk, (int)kp.nbf_pad, (double*)cocc, (double*)sign);
    else
        hipLaunchKernelGGL(k_prep_cocc_idx<float>, g, dim3(256), 0, st, vecs, (int)nbf, idx, lam, (int)ncol,
                           (int)col_off, (int)kp.nk, (int)kp.nbf_pad, (float*)cocc, (float*)sign);
    return hipGetLastError();
}

hipError_t launch_prep_factor(hipStream_t st, const double* f, size_t nbf, size_t fs, const size_t* ncol, int nspin,
                              const KPlan& kp, double* cocc, double* sign) {
    const size_t n = kp.nbf_pad * kp.nk;
    hipLaunchKernelGGL(k_prep_factor, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, f, (int)nbf, fs, (int)ncol[0],
                       nspin == 2 ? (int)ncol[1] : 0, (int)kp.col_off[1], (int)kp.nk, (int)kp.nbf_pad, cocc, sign);
    return hipGetLastError();
}

hipError_t launch_khalf(hipStream_t st, int prec, const void* b, size_t ldb, size_t nbf, size_t P0, size_t Pc,
                        const KPlan& kp, const void* cocc, void* m) {
    if (prec == RJK_PREC_FP64)
        return khalf_t<double>(st, (const double*)b, ldb, nbf, P0, Pc, kp, (const double*)cocc, (double*)m);
    return khalf_t<float>(st, (const float*)b, ldb, nbf, P0, Pc, kp, (const float*)cocc, (float*)m);
}

hipError_t launch_ksyrk(hipStream_t st, int prec, const void* m, size_t nbf, size_t Pc, const KPlan& kp, int nspin,
                        const void* sign, int beta, double* kpart) {
    if (prec == RJK_PREC_FP64)
        return ksyrk_t<double>(st, (const double*)m, nbf, Pc, kp, nspin, (const double*)sign, beta, kpart);
    return ksyrk_t<float>(st, (const float*)m, nbf, Pc, kp, nspin, (const float*)sign, beta, kpart);
}

hipError_t launch_kreduce(hipStream_t st, const double* kpart, const KPlan& kp, int nspin, size_t nbf, double scale,
                          double* vk) {
    size_t npair = nbf * (nbf + 1) / 2;
    hipLaunchKernelGGL(k_kreduce, dim3((unsigned)((npair + kRedPairs - 1) / kRedPairs), (unsigned)nspin),
                       dim3(kRedPairs * kRedGroups), 0, st, kpart, (int)kp.nslot, nspin, kp.nbf_pad * kp.nbf_pad,
                       (int)kp.nbf_pad, npair, scale, vk);
    return hipGetLastError();
}

}  // namespace rjk
