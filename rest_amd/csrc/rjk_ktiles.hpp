// rjk_ktiles.hpp — the K tiles (half-transform and SYRK) as device functions,
// shared by the single-problem kernels (rjk_k.hip) and the grouped persistent
// kernels of a batch of problems (rjk_batch.hip).
//
// MFMA: v_mfma_f64_16x16x4f64.  Lane l supplies A[l%16][l/16] and
// B[l/16][l%16]; register r of lane l receives D[l/16 + 4r][l%16] (probed on
// gfx950).  Both tiles put the memory-contiguous index (μ) on the D column
// so that 16 consecutive lanes store 128 contiguous bytes.
#pragma once
#include "rjk_internal.hpp"

namespace rjk {
namespace kt {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int kBlock = 256;           // 4 waves
constexpr int TK = kTileK;            // 16
// LDS row padding (elements).  FP64: rows of 128 + 2 (or 64 + 2) doubles put the 16 rows that
// one transposed stash instruction writes (one element each, 16 lanes at a time) on 16 distinct
// 4-bank groups, and the 16 consecutive doubles of a fragment read on consecutive banks; a pad of
// 4 leaves rows k and k + 8 on the same banks.  FP32 keeps 4.
template <typename T> struct Pad { static constexpr int v = sizeof(T) == 8 ? 2 : 4; };
constexpr int kXcd = 8;               // MI355X: 8 XCDs, work-groups dealt round-robin by linear id

__device__ inline size_t tri(size_t j) { return j * (j + 1) / 2; }

// A device pointer read from a table in memory (not a kernel argument) is a flat pointer to the
// compiler, and flat loads count against the LDS wait counter as well as the vector-memory one,
// so every LDS wait of a pipelined tile would also wait for the next block's loads.  glb() gives
// such a pointer the global address space; the tiles below take their pointers as template types,
// so these accesses stay global loads and stores.
#define RJK_GLB __attribute__((address_space(1)))
template <typename T> __device__ __forceinline__ RJK_GLB T* glb(T* p) { return (RJK_GLB T*)p; }

// Rotation of a work-group's rows over its waves.  Work-groups that share a CU are about 32 apart in
// the XCD-local order, so neighbours on a CU get different rotations and the waves that skip padding
// or below-diagonal fragments do not all sit on the same SIMD.
__device__ __forceinline__ int rotation(int kq) { return (kq + kq / 32) & 3; }

// One 16x16x4 MFMA per element type.  Lane l supplies A[l%16][l/16] and
// B[l/16][l%16]; register r of lane l holds D[row(l, r)][l%16] (probed on
// gfx950: FP64 interleaves rows by 4, FP32 keeps 4 consecutive rows).
template <typename T> struct Mma;
template <> struct Mma<double> {
    using acc_t = d4;
    __device__ static acc_t zero() { return d4{0.0, 0.0, 0.0, 0.0}; }
    __device__ static acc_t op(double a, double b, acc_t c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    __device__ static int row(int lane, int r) { return (lane >> 4) + 4 * r; }
};
template <> struct Mma<float> {
    using acc_t = f4;
    __device__ static acc_t zero() { return f4{0.f, 0.f, 0.f, 0.f}; }
    __device__ static acc_t op(float a, float b, acc_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    __device__ static int row(int lane, int r) { return 4 * (lane >> 4) + r; }
};

// upper tile pair (tm <= tn) of packed tile index t
__device__ inline void upper_tile(size_t t, size_t* tm, size_t* tn) {
    size_t n = (size_t)((sqrt(8.0 * (double)t + 1.0) - 1.0) * 0.5);
    while (tri(n) > t) --n;
    while (tri(n + 1) <= t) ++n;
    *tn = n;
    *tm = t - tri(n);
}

// What bounds these tiles: on gfx950 the FP64 and FP32 MFMAs run at the rate of the vector unit and
// keep it busy, so every other vector instruction of any wave on that SIMD costs about 5 cycles of
// MFMA time (measured: 8 FP64 MFMAs alone 523 cycles a wave, with 64 integer instructions 859; FP32
// 274 and 595; BF16 MFMAs overlap with them).  The tiles therefore address memory through wave-
// uniform bases (scalar registers) plus lane offsets that stay the same for the whole tile, and
// choose the way an operand is read per k-block by scalar branches: 20-40 vector instructions per
// k-block of 16 (32-64 MFMAs) in place of about 250.
template <typename T, int N> struct VecOf {
    typedef T raw __attribute__((ext_vector_type(N)));
    typedef T type __attribute__((ext_vector_type(N), aligned(sizeof(T))));   // element alignment
};
template <typename T> __device__ __forceinline__ RJK_GLB const T* as_glb(const T* p) { return (RJK_GLB const T*)p; }
template <typename T> __device__ __forceinline__ RJK_GLB const T* as_glb(RJK_GLB const T* p) { return p; }
// N elements at base (uniform) + off bytes (per lane)
template <typename T, int N>
__device__ __forceinline__ typename VecOf<T, N>::raw ldv(RJK_GLB const T* base, unsigned off) {
    return *(RJK_GLB const typename VecOf<T, N>::type*)((RJK_GLB const char*)base + off);
}

// ---------------------------------------------------------------------------
// Stage 1: M'[P][c][μ] = Σ_ν Bsym_P[μ,ν] C'[ν][c], one (μ-tile, c-tile) of one
//   auxiliary column: 64·FM μ rows on 4 waves, 16·FN columns c.  The caller picks
//   FN so that few columns are padding; a wave whose 16·FM rows all lie beyond nbf
//   skips its MFMAs, and `rot` rotates the rows over the waves so that the skipped
//   ones fall on different SIMDs.  Rows μ >= nbf of M' are left unwritten or hold
//   finite padding: nothing reads them into an output.  Software pipeline: the next
//   k-block is fetched into registers while the MFMAs consume the current one from
//   LDS (double-buffered, one barrier per k-block).  Sums run over ν in ascending
//   order whatever the tile, so M' does not depend on FM and FN.
//
//   Reading the packed column (element (i <= j) at tri(j) + i):
//     blocks left of the tile's diagonal range (ν < mu0): along ν, two elements a lane at
//       offsets fixed for the tile, the base moving by 16 elements a block;
//     blocks beyond it (ν >= mu0 + 64 FM): row ν is contiguous in μ, one row per wave
//       instruction at a scalar base;
//     the diagonal blocks and a partial last block: element by element, mirrored and masked.
// ---------------------------------------------------------------------------
template <typename T, int FM, int FN, typename BP, typename CP, typename MP>
__device__ __forceinline__ void khalf_tile(BP __restrict__ bcol_, int nbf, int mu0, int c0, CP __restrict__ cocc_,
                                           int nk, int ldm, MP __restrict__ mP, int rot) {
    using MM = Mma<T>;
    constexpr int TM = 64 * FM, TN = 16 * FN, NA = 4 * FM;
    constexpr int VB = 16 / (int)sizeof(T), PRB = TN / VB, NPB = TK * PRB, NB = (NPB + kBlock - 1) / kBlock;
    using VA = typename VecOf<T, FM>::raw;
    using V2 = typename VecOf<T, 2>::raw;
    using VBt = typename VecOf<T, VB>::raw;
    __shared__ __align__(16) T As[2][TK][TM + Pad<T>::v];
    __shared__ __align__(16) T Bs[2][TK][TN + Pad<T>::v];
    const auto bcol = as_glb(bcol_);
    const auto cocc = as_glb(cocc_);
    const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), ws = (wave + rot) & 3;
    T ra[NA];
    VBt rb[NB];
    unsigned live = 0;   // element-wise blocks: bit r set when element r lies inside nbf × nbf
    if (mu0 >= nbf) return;   // a tile of padding rows only (nbf_pad beyond the tile grid); uniform

    // lane offsets (bytes), fixed for the tile
    unsigned offd[2 * FM], offb[NB];
#pragma unroll
    for (int r = 0; r < 2 * FM; ++r) {
        const int mu = min(mu0 + (tid >> 3) + 32 * r, nbf - 1);
        offd[r] = (unsigned)((tri((size_t)mu) - tri((size_t)mu0) + (tid & 7) * 2) * sizeof(T));
    }
#pragma unroll
    for (int r = 0; r < NB; ++r) {
        const int e = min(tid + r * kBlock, NPB - 1);
        offb[r] = (unsigned)(((e / PRB) * nk + (e % PRB) * VB) * sizeof(T));
    }
    const unsigned offa = lane * FM * sizeof(T);

    enum { BELOW, ABOVE, MIXED };
    auto fetch = [&](auto kind, int nu0) {
        if constexpr (kind() == BELOW) {
            const auto p = bcol + tri((size_t)mu0) + nu0;
#pragma unroll
            for (int r = 0; r < 2 * FM; ++r) {
                const V2 v = ldv<T, 2>(p, offd[r]);
                ra[2 * r] = v[0];
                ra[2 * r + 1] = v[1];
            }
        } else if constexpr (kind() == ABOVE) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const VA v = ldv<T, FM>(bcol + tri((size_t)(nu0 + wave + 4 * r)) + mu0, offa);
#pragma unroll
                for (int q = 0; q < FM; ++q) ra[r * FM + q] = v[q];
            }
        } else {
            live = 0;
#pragma unroll
            for (int r = 0; r < NA; ++r) {
                const int e = tid + r * kBlock, mu = mu0 + e % TM, nu = nu0 + e / TM;
                const int lo = mu < nu ? mu : nu, hi = mu < nu ? nu : mu;
                const bool ok = hi < nbf;
                live |= (unsigned)ok << r;
                ra[r] = bcol[ok ? tri((size_t)hi) + lo : 0];
            }
        }
        const auto q = cocc + (size_t)nu0 * nk + c0;   // C' rows are zero-padded beyond nbf
#pragma unroll
        for (int r = 0; r < NB; ++r) rb[r] = ldv<T, VB>(q, offb[r]);
    };
    auto stash = [&](auto kind, int buf) {
        if constexpr (kind() == BELOW) {
#pragma unroll
            for (int r = 0; r < 2 * FM; ++r) {
                As[buf][(tid & 7) * 2][(tid >> 3) + 32 * r] = ra[2 * r];
                As[buf][(tid & 7) * 2 + 1][(tid >> 3) + 32 * r] = ra[2 * r + 1];
            }
        } else if constexpr (kind() == ABOVE) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                VA v;
#pragma unroll
                for (int q = 0; q < FM; ++q) v[q] = ra[r * FM + q];
                *(VA*)&As[buf][wave + 4 * r][lane * FM] = v;
            }
        } else {
#pragma unroll
            for (int r = 0; r < NA; ++r) {
                const int e = tid + r * kBlock;
                As[buf][e / TM][e % TM] = ((live >> r) & 1u) ? ra[r] : T(0);
            }
        }
#pragma unroll
        for (int r = 0; r < NB; ++r) {
            const int e = tid + r * kBlock;
            if ((r + 1) * kBlock <= NPB || e < NPB) *(VBt*)&Bs[buf][e / PRB][(e % PRB) * VB] = rb[r];
        }
    };

    typename MM::acc_t acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = MM::zero();
    const int mrow = ws * 16 * FM;
    const bool act = mu0 + mrow < nbf;   // wave-uniform
    auto compute = [&](int cur) {
        if (!act) return;
#pragma unroll
        for (int kk = 0; kk < TK; kk += 4) {
            T bmu[FM], ac[FN];
#pragma unroll
            for (int i = 0; i < FM; ++i) bmu[i] = As[cur][kk + g][mrow + i * 16 + l16];
#pragma unroll
            for (int j = 0; j < FN; ++j) ac[j] = Bs[cur][kk + g][j * 16 + l16];
            // D[c][μ] = Σ_ν C'[ν][c] Bsym[ν][μ]
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j) acc[i][j] = MM::op(ac[j], bmu[i], acc[i][j]);
        }
    };

    // k-blocks [0, e0) below the diagonal range, [e0, e1) across it, [e1, e2) above, [e2, nkb) the partial last
    const int nkb = (nbf + TK - 1) / TK;
    const int e0 = mu0 / TK, e1 = min(nkb, (mu0 + TM) / TK), e2 = max(e1, nbf / TK);
    struct KB { __device__ constexpr int operator()() const { return BELOW; } };
    struct KA { __device__ constexpr int operator()() const { return ABOVE; } };
    struct KX { __device__ constexpr int operator()() const { return MIXED; } };
    int kb = 0;
    auto run = [&](auto kind, int end) {   // blocks up to `end` are of this kind; block kb is in LDS
        for (; kb + 1 < end; ++kb) {
            fetch(kind, (kb + 1) * TK);
            compute(kb & 1);
            stash(kind, (kb + 1) & 1);
            __syncthreads();
        }
    };
    if (e0 > 0) {
        fetch(KB(), 0);
        stash(KB(), 0);
    } else {
        fetch(KX(), 0);
        stash(KX(), 0);
    }
    __syncthreads();
    run(KB(), e0);
    run(KX(), e1);
    run(KA(), e2);
    run(KX(), nkb);
    compute(kb & 1);
    __syncthreads();   // the persistent callers start their next tile in the same LDS

    if (!act) return;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            const int mu = mu0 + mrow + i * 16 + l16, cb = c0 + j * 16;
#pragma unroll
            for (int r = 0; r < 4; ++r) mP[(size_t)(cb + MM::row(lane, r)) * ldm + mu] = acc[i][j][r];
        }
}

// ---------------------------------------------------------------------------
// Stage 2: Kpart (+)= Σ_{P,c} M'[P][c][μ] sign_c M'[P][c][ν] over the upper tiles
//   (mu0 <= nu0) of 64·FB × 64·FB, split-K over P.  Wave w owns 16·FB columns ν and
//   every row μ of the tile; in a diagonal tile it computes only the μ groups up to its
//   own (10 of 16 groups), and a wave whose columns all lie beyond nbf computes nothing
//   (`rot` as in stage 1).  Same pipeline as stage 1 over the flattened (P, 16-column block) index;
//   the rows of M' are wave-uniform, so every load is one row at a scalar base.  Signs
//   are looked at once per tile and applied while staging only where one is negative.
//   Accumulation in the MFMA type, partial tiles kept in FP64.
// ---------------------------------------------------------------------------
struct SyrkCols {
    int off[2], cnt[2];
};

template <typename T, int FB, bool DIAG, typename MP, typename SP, typename KP>
__device__ __forceinline__ void ksyrk_body(MP m, int ldm, int nk, int nbf, int mu0, int nu0, int cb, int ncb, int Pb,
                                           int Pe, SP sign, int beta, KP kp, int ws, bool neg, T* __restrict__ lds) {
    using MM = Mma<T>;
    constexpr int FA = 4 * FB, Tt = 64 * FB, LD = Tt + Pad<T>::v;
    using VL = typename VecOf<T, FB>::raw;
    const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    auto As = [&](int buf, int k) { return lds + (buf * TK + k) * LD; };
    auto Bs = [&](int buf, int k) { return lds + ((2 + buf) * TK + k) * LD; };
    const int nq = (Pe > Pb ? Pe - Pb : 0) * ncb;
    const unsigned off = lane * FB * sizeof(T);
    VL ra[4], rb[4];
    T rs[4];
    int fP = Pb, fc = 0;   // (P, block) of the next fetch
    auto fetch = [&]() {
        const auto base = m + ((size_t)fP * nk + cb + fc * TK + wave) * ldm;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if constexpr (!DIAG) ra[r] = ldv<T, FB>(base + (size_t)(4 * r) * ldm + mu0, off);
            rb[r] = ldv<T, FB>(base + (size_t)(4 * r) * ldm + nu0, off);
        }
        if (neg) {
#pragma unroll
            for (int r = 0; r < 4; ++r) rs[r] = sign[cb + fc * TK + wave + 4 * r];
        }
        if (++fc == ncb) {
            fc = 0;
            ++fP;
        }
    };
    // a diagonal tile stages its rows once, and a second time with the signs where one is negative
    auto stash = [&](int buf) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if constexpr (DIAG) *(VL*)(As(buf, wave + 4 * r) + lane * FB) = rb[r];
            else *(VL*)(As(buf, wave + 4 * r) + lane * FB) = ra[r];
            if (!DIAG || neg) *(VL*)(Bs(buf, wave + 4 * r) + lane * FB) = neg ? rb[r] * rs[r] : rb[r];
        }
    };
    typename MM::acc_t acc[FA][FB];
#pragma unroll
    for (int i = 0; i < FA; ++i)
#pragma unroll
        for (int j = 0; j < FB; ++j) acc[i][j] = MM::zero();
    const int ncol = ws * 16 * FB;
    const bool act = nu0 + ncol < nbf;
    const int bsel = (!DIAG || neg) ? 2 * TK * LD : 0;   // where the ν operand lies
    auto compute = [&](int cur) {
        if (!act) return;
        const T* __restrict__ a0 = As(cur, g) + l16;
        const T* __restrict__ b0 = As(cur, g) + bsel + ncol + l16;
        // D[ν][μ] = Σ_k sign_k M'[k][ν] M'[k][μ]
        if constexpr (DIAG) {
            T anu[TK / 4][FB];
#pragma unroll
            for (int kk = 0; kk < TK; kk += 4)
#pragma unroll
                for (int j = 0; j < FB; ++j) anu[kk / 4][j] = b0[kk * LD + j * 16];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if (q > ws) break;   // groups of FB fragments; those right of the wave's own are below the diagonal
#pragma unroll
                for (int kk = 0; kk < TK; kk += 4) {
                    T bmu[FB];
#pragma unroll
                    for (int i = 0; i < FB; ++i) bmu[i] = a0[kk * LD + (q * FB + i) * 16];
#pragma unroll
                    for (int i = 0; i < FB; ++i)
#pragma unroll
                        for (int j = 0; j < FB; ++j)
                            acc[q * FB + i][j] = MM::op(anu[kk / 4][j], bmu[i], acc[q * FB + i][j]);
                }
            }
        } else {
#pragma unroll
            for (int kk = 0; kk < TK; kk += 4) {
                T bmu[FA], anu[FB];
#pragma unroll
                for (int j = 0; j < FB; ++j) anu[j] = b0[kk * LD + j * 16];
#pragma unroll
                for (int i = 0; i < FA; ++i) bmu[i] = a0[kk * LD + i * 16];
#pragma unroll
                for (int i = 0; i < FA; ++i)
#pragma unroll
                    for (int j = 0; j < FB; ++j) acc[i][j] = MM::op(anu[j], bmu[i], acc[i][j]);
            }
        }
    };
    if (nq > 0) {
        fetch();
        stash(0);
    }
    __syncthreads();
    for (int q = 0; q + 1 < nq; ++q) {
        fetch();
        compute(q & 1);
        stash((q + 1) & 1);
        __syncthreads();
    }
    if (nq > 0) compute((nq - 1) & 1);
    __syncthreads();   // the persistent callers start their next tile in the same LDS
    if (!act) return;
#pragma unroll
    for (int i = 0; i < FA; ++i) {
        if (DIAG && i / FB > ws) break;
#pragma unroll
        for (int j = 0; j < FB; ++j) {
            const int mu = mu0 + i * 16 + l16, nb = nu0 + ncol + j * 16;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const auto dst = kp + (size_t)(nb + MM::row(lane, r)) * ldm + mu;
                double v = (double)acc[i][j][r];
                if (beta) v += *dst;
                *dst = v;
            }
        }
    }
}

template <typename T, int FB, typename MP, typename SP, typename KP>
__device__ __forceinline__ void ksyrk_tile(MP __restrict__ m, int ldm, int nk, int nbf, int mu0, int nu0, int cb,
                                           int ncb, int Pb, int Pe, SP __restrict__ sign, int beta,
                                           KP __restrict__ kp, int rot) {
    constexpr int LD = 64 * FB + Pad<T>::v;
    __shared__ __align__(16) T lds[4 * TK * LD];
    const int ws = (__builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6) + rot) & 3;
    if (nu0 >= nbf) return;   // padding columns only (uniform)
    int any = 0;
    for (int c = threadIdx.x; c < ncb * TK; c += kBlock) any |= sign[cb + c] < T(0);
    const bool neg = __syncthreads_or(any) != 0;
    const auto mg = as_glb(m);
    if (mu0 == nu0)
        ksyrk_body<T, FB, true>(mg, ldm, nk, nbf, mu0, nu0, cb, ncb, Pb, Pe, sign, beta, kp, ws, neg, lds);
    else
        ksyrk_body<T, FB, false>(mg, ldm, nk, nbf, mu0, nu0, cb, ncb, Pb, Pe, sign, beta, kp, ws, neg, lds);
}


}  // namespace kt
}  // namespace rjk
