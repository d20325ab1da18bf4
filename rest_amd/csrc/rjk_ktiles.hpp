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
// LDS row padding (elements).  A fragment read takes 16 consecutive elements of each of 4 rows.
// FP64 serves one row a cycle whatever their distance; 2 elements keep the transposed stash of
// blocks left of the diagonal off one bank.  FP32 serves two rows a cycle, free of conflicts when
// the row length is an odd multiple of 16.
template <typename T> constexpr int row_pad(int n) { return sizeof(T) == 8 ? 2 : ((n / 16) % 2 ? 0 : 16); }
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
// N elements at base (uniform) + off bytes (per lane).  The empty asm keeps the widening of `off` next
// to the load, which is what lets it use the scalar-base form (a widening hoisted out of the loop
// costs a 64-bit vector addition a load).
template <typename T, int N>
__device__ __forceinline__ typename VecOf<T, N>::raw ldv(RJK_GLB const T* base, unsigned& off) {
    asm("" : "+v"(off));
    return *(RJK_GLB const typename VecOf<T, N>::type*)((RJK_GLB const char*)base + off);
}

// an LDS buffer as a compile-time number, so that it is part of an instruction's offset
template <int N> struct Buf { static constexpr int n = N; };

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
//     the diagonal blocks: element by element, mirrored by one select on wave-uniform rows;
//     a partial last block: element by element, mirrored and masked.
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
    __shared__ __align__(16) T As[2][TK][TM + row_pad<T>(TM)];
    __shared__ __align__(16) T Bs[2][TK][TN + (sizeof(T) == 8 ? 0 : row_pad<T>(TN))];   // FP64: 3 work-groups a CU at FN = 5
    const auto bcol = as_glb(bcol_);
    const auto cocc = as_glb(cocc_);
    const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), ws = (wave + rot) & 3;
    T ra[NA];
    VBt rb[NB];
    unsigned live = 0;   // partial last block: bit r set when element r lies inside nbf × nbf
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
    unsigned offa = lane * FM * sizeof(T);
    // diagonal blocks: row h = max, column l = min of the two tile-relative indices lies h·mu0 + tri(h) + l
    // beyond element (mu0, mu0); a thread keeps one μ, ν is wave-uniform
    const int mt = min(tid % TM, nbf - 1 - mu0);
    const unsigned offm = (unsigned)(mt * sizeof(T)), offr = (unsigned)((mt * mu0 + mt * (mt + 1) / 2) * sizeof(T));

    enum { BELOW, DIAG, ABOVE, TAIL };
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
        } else if constexpr (kind() == DIAG) {
            const auto p = bcol + tri((size_t)mu0) + mu0;
#pragma unroll
            for (int r = 0; r < NA; ++r) {
                const int x = nu0 - mu0 + wave * 64 / TM + r * (kBlock / TM);   // tile-relative ν, uniform
                unsigned o = x <= mt ? offr + (unsigned)(x * sizeof(T))
                                     : offm + (unsigned)((x * mu0 + x * (x + 1) / 2) * sizeof(T));
                ra[r] = ldv<T, 1>(p, o)[0];
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
    T* const sa_below = &As[0][(tid & 7) * 2][tid >> 3];
    T* const sa_above = &As[0][wave][lane * FM];
    constexpr int LA = TM + row_pad<T>(TM), LB = TN + (sizeof(T) == 8 ? 0 : row_pad<T>(TN));
    auto stash = [&](auto kind, int buf) {
        if constexpr (kind() == BELOW) {
#pragma unroll
            for (int r = 0; r < 2 * FM; ++r) {
                sa_below[buf * TK * LA + 32 * r] = ra[2 * r];
                sa_below[buf * TK * LA + LA + 32 * r] = ra[2 * r + 1];
            }
        } else if constexpr (kind() == ABOVE) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                VA v;
#pragma unroll
                for (int q = 0; q < FM; ++q) v[q] = ra[r * FM + q];
                *(VA*)(sa_above + (buf * TK + 4 * r) * LA) = v;
            }
        } else {
#pragma unroll
            for (int r = 0; r < NA; ++r) {
                const int e = tid + r * kBlock;
                As[buf][e / TM][e % TM] = (kind() == DIAG || ((live >> r) & 1u)) ? ra[r] : T(0);
            }
        }
#pragma unroll
        for (int r = 0; r < NB; ++r) {
            const int e = tid + r * kBlock;
            if ((r + 1) * kBlock <= NPB || e < NPB) *(VBt*)(&Bs[0][e / PRB][(e % PRB) * VB] + buf * TK * LB) = rb[r];
        }
    };

    typename MM::acc_t acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = MM::zero();
    const int mrow = ws * 16 * FM;
    const bool act = mu0 + mrow < nbf;   // wave-uniform
    const T* const fa = &As[0][g][mrow + l16];
    const T* const fb = &Bs[0][g][l16];
    auto compute = [&](int cur) {
        if (!act) return;
#pragma unroll
        for (int kk = 0; kk < TK; kk += 4) {
            T bmu[FM], ac[FN];
#pragma unroll
            for (int i = 0; i < FM; ++i) bmu[i] = fa[(cur * TK + kk) * LA + i * 16];
#pragma unroll
            for (int j = 0; j < FN; ++j) ac[j] = fb[(cur * TK + kk) * LB + j * 16];
            // D[c][μ] = Σ_ν C'[ν][c] Bsym[ν][μ]
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j) acc[i][j] = MM::op(ac[j], bmu[i], acc[i][j]);
        }
    };

    // k-blocks [0, e0) below the diagonal range, [e0, e1) across it, [e1, e2) above, [e2, nkb) the partial last
    const int nkb = (nbf + TK - 1) / TK, e2 = nbf / TK;
    const int e0 = mu0 / TK, e1 = min(e2, (mu0 + TM) / TK);
    struct KB { __device__ constexpr int operator()() const { return BELOW; } };
    struct KD { __device__ constexpr int operator()() const { return DIAG; } };
    struct KA { __device__ constexpr int operator()() const { return ABOVE; } };
    struct KT { __device__ constexpr int operator()() const { return TAIL; } };
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
    } else if (e1 > 0) {
        fetch(KD(), 0);
        stash(KD(), 0);
    } else {
        fetch(KT(), 0);
        stash(KT(), 0);
    }
    __syncthreads();
    run(KB(), e0);
    run(KD(), e1);
    run(KA(), e2);
    run(KT(), nkb);
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
//   (mu0 <= nu0) of 32·F × 32·F, split-K over P, 2 × 2 waves of F × F fragments.  In a
//   diagonal tile the wave below the diagonal computes nothing (the two on it all of
//   theirs), nor do waves beyond nbf (`rot` as in stage 1).
//   Same pipeline as stage 1 over the flattened (P, 16-column block) index: lane offsets
//   within a k-block's 16 rows are fixed, the base moves by scalar arithmetic.  A diagonal
//   tile stages its rows once for both operands.  Signs are looked at once per tile and
//   applied while staging only where one is negative.  Accumulation in the MFMA type,
//   partial tiles kept in FP64.
//   Loads run two k-blocks ahead in two register sets, so that a miss to HBM is covered also with
//   two waves a SIMD; with the LDS buffers as compile-time offsets a k-block costs no vector
//   instruction beside its MFMAs.  FP64 inner rate (k-blocks from L2, 2 work-groups a CU): F = 4
//   71 TFLOP/s, F = 2 66 (F = 3 on three work-groups 65; one block ahead and dynamic buffers 67, 62, 65).
// ---------------------------------------------------------------------------
struct SyrkCols {
    int off[2], cnt[2];
};

template <typename T, int F, bool DIAG, typename MP, typename SP, typename KP>
__device__ __forceinline__ void ksyrk_body(MP m, int ldm, int nk, int nbf, int mu0, int nu0, int cb, int ncb, int Pb,
                                           int Pe, SP sign, int beta, KP kp, int ws, bool neg, T* __restrict__ lds) {
    using MM = Mma<T>;
    constexpr int Tt = 32 * F, LD = Tt + row_pad<T>(Tt);
    constexpr int VB = 16 / (int)sizeof(T) < F * 32 * TK / kBlock ? 16 / (int)sizeof(T) : F * 32 * TK / kBlock;
    constexpr int PR = Tt / VB, NL = TK * PR / kBlock;   // pieces a row, pieces a thread
    static_assert(NL * kBlock == TK * PR, "load shape");
    using VL = typename VecOf<T, VB>::raw;
    const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, g = lane >> 4;
    // LDS: μ operand of buffers 0 and 1, then the ν operand of both
    constexpr int kB = 2 * TK * LD;
    const int nq = (Pe > Pb ? Pe - Pb : 0) * ncb;
    unsigned off[NL];
#pragma unroll
    for (int r = 0; r < NL; ++r) {
        const int e = tid + r * kBlock;
        off[r] = (unsigned)(((e / PR) * ldm + (e % PR) * VB) * sizeof(T));
    }
    // two register sets: block q + 2 is under way while block q + 1 waits to be staged
    VL ra0[NL], rb0[NL], ra1[NL], rb1[NL];
    int fP = Pb, fc = 0, fq = 0;   // (P, block) of the next fetch; past the last block it repeats that one
    auto fetch = [&](VL (&ra)[NL], VL (&rb)[NL]) {
        const auto base = m + ((size_t)fP * nk + cb + fc * TK) * ldm;
#pragma unroll
        for (int r = 0; r < NL; ++r) {
            if constexpr (!DIAG) ra[r] = ldv<T, VB>(base + mu0, off[r]);
            rb[r] = ldv<T, VB>(base + nu0, off[r]);
        }
        if (++fq < nq && ++fc == ncb) {
            fc = 0;
            ++fP;
        }
    };
    T* sw[NL];
#pragma unroll
    for (int r = 0; r < NL; ++r) sw[r] = lds + ((tid + r * kBlock) / PR) * LD + ((tid + r * kBlock) % PR) * VB;
    int sc = 0;   // column block of the next stash
    auto stash = [&](auto buf, VL (&ra)[NL], VL (&rb)[NL]) {
        constexpr int o = decltype(buf)::n * TK * LD;
#pragma unroll
        for (int r = 0; r < NL; ++r) {
            if constexpr (DIAG) *(VL*)(sw[r] + o) = rb[r];
            else *(VL*)(sw[r] + o) = ra[r];
            if (!DIAG && !neg) *(VL*)(sw[r] + kB + o) = rb[r];
        }
        if (neg) {   // signed columns (rare): the signs are read here
#pragma unroll
            for (int r = 0; r < NL; ++r)
                *(VL*)(sw[r] + kB + o) = rb[r] * (T)sign[cb + sc * TK + (tid + r * kBlock) / PR];
            if (++sc == ncb) sc = 0;
        }
    };
    typename MM::acc_t acc[F][F];
#pragma unroll
    for (int i = 0; i < F; ++i)
#pragma unroll
        for (int j = 0; j < F; ++j) acc[i][j] = MM::zero();
    const int mrow = (ws & 1) * 16 * F, ncol = (ws >> 1) * 16 * F;
    const bool act = nu0 + ncol < nbf && mu0 + mrow < nbf && !(DIAG && mrow > ncol);
    const T* const fa = lds + g * LD + mrow + l16;
    const T* const fb = lds + g * LD + ncol + l16 + ((!DIAG || neg) ? kB : 0);
    auto compute = [&](auto cur_) {
        constexpr int cur = decltype(cur_)::n;
        if (!act) return;
        // D[ν][μ] = Σ_k sign_k M'[k][ν] M'[k][μ]
#pragma unroll
        for (int kk = 0; kk < TK; kk += 4) {
            T bmu[F], anu[F];
#pragma unroll
            for (int j = 0; j < F; ++j) anu[j] = fb[(cur * TK + kk) * LD + j * 16];
#pragma unroll
            for (int i = 0; i < F; ++i) bmu[i] = fa[(cur * TK + kk) * LD + i * 16];
#pragma unroll
            for (int i = 0; i < F; ++i)
#pragma unroll
                for (int j = 0; j < F; ++j) acc[i][j] = MM::op(anu[j], bmu[i], acc[i][j]);
        }
    };
    if (nq > 0) {
        fetch(ra0, rb0);
        fetch(ra1, rb1);
        stash(Buf<0>(), ra0, rb0);
        fetch(ra0, rb0);
    }
    __syncthreads();
    for (int q = 0; q < nq; q += 2) {   // an odd last block leaves buffer 1 unused
        compute(Buf<0>());
        stash(Buf<1>(), ra1, rb1);
        fetch(ra1, rb1);
        __syncthreads();
        if (q + 1 < nq) compute(Buf<1>());
        stash(Buf<0>(), ra0, rb0);
        fetch(ra0, rb0);
        __syncthreads();
    }
    __syncthreads();   // the persistent callers start their next tile in the same LDS
    if (!act) return;
#pragma unroll
    for (int i = 0; i < F; ++i)
#pragma unroll
        for (int j = 0; j < F; ++j) {
            const int mu = mu0 + mrow + i * 16 + l16, nb = nu0 + ncol + j * 16;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const auto dst = kp + (size_t)(nb + MM::row(lane, r)) * ldm + mu;
                double v = (double)acc[i][j][r];
                if (beta) v += *dst;
                *dst = v;
            }
        }
}

template <typename T, int F, typename MP, typename SP, typename KP>
__device__ __forceinline__ void ksyrk_tile(MP __restrict__ m, int ldm, int nk, int nbf, int mu0, int nu0, int cb,
                                           int ncb, int Pb, int Pe, SP __restrict__ sign, int beta,
                                           KP __restrict__ kp, int rot) {
    constexpr int LD = 32 * F + row_pad<T>(32 * F);
    __shared__ __align__(16) T lds[4 * TK * LD];
    const int ws = (__builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6) + rot) & 3;
    if (nu0 >= nbf) return;   // padding columns only (uniform)
    int any = 0;
    for (int c = threadIdx.x; c < ncb * TK; c += kBlock) any |= sign[cb + c] < T(0);
    const bool neg = __syncthreads_or(any) != 0;
    const auto mg = as_glb(m);
    if (mu0 == nu0)
        ksyrk_body<T, F, true>(mg, ldm, nk, nbf, mu0, nu0, cb, ncb, Pb, Pe, sign, beta, kp, ws, neg, lds);
    else
        ksyrk_body<T, F, false>(mg, ldm, nk, nbf, mu0, nu0, cb, ncb, Pb, Pe, sign, beta, kp, ws, neg, lds);
}


}  // namespace kt
}  // namespace rjk
