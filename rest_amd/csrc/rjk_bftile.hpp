// rjk_bftile.hpp — one work-group tile of D[x][y] += Σ_k X[x][k] Y[y][k] on the BF16
// matrix cores with operands split into S planes (both operands k-contiguous rows).
//
// Plane products: the pairs (a, b) with a + b < S, one v_mfma_f32_16x16x32_bf16 each
// (lane l supplies A[l%16][8(l/16)+i] = X and B[8(l/16)+i][l%16] = Yᵀ; register r of
// lane l receives D[4(l/16)+r][l%16], probed on gfx950).  Accumulation in FP32.
//
// A work-group of WX × WY waves covers WGX × WGY outputs; wave (wx, wy) owns
// FX × FY fragments of 16 × 16.  Per k-block of TK (32 or 64), every wave moves fragments of
// both operands from global memory into registers, then into LDS; the next k-block's
// global loads are in flight while the MFMAs run.  LDS holds the fragments as memory does, so
// that both its writes and its reads are 64 pieces in a row, free of bank conflicts.
#pragma once
#include <hip/hip_runtime.h>

namespace rjk {
namespace bft {

typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef unsigned int u2 __attribute__((ext_vector_type(2)));
typedef unsigned int u4 __attribute__((ext_vector_type(4)));

constexpr int KM = 32;        // one MFMA deep

// plane pair (X plane, Y plane) of product p
template <int S> __device__ constexpr int pa(int p);
template <int S> __device__ constexpr int pb(int p);
template <> __device__ constexpr int pa<1>(int) { return 0; }
template <> __device__ constexpr int pb<1>(int) { return 0; }
template <> __device__ constexpr int pa<2>(int p) { return p == 2 ? 1 : 0; }
template <> __device__ constexpr int pb<2>(int p) { return p == 1 ? 1 : 0; }
template <> __device__ constexpr int pa<3>(int p) { return p == 2 || p == 4 ? 1 : (p == 5 ? 2 : 0); }
template <> __device__ constexpr int pb<3>(int p) { return p == 1 || p == 4 ? 1 : (p == 3 ? 2 : 0); }
template <int S> constexpr int npairs() { return S * (S + 1) / 2; }

template <int S_, int WGX_, int WGY_, int WX_, int WY_, int TK_ = 32>
struct Cfg {
    static constexpr int S = S_, WGX = WGX_, WGY = WGY_, WX = WX_, WY = WY_, TK = TK_;
    static constexpr int NT = WX * WY * 64;
    static constexpr int FX = WGX / WX / 16, FY = WGY / WY / 16;
    static constexpr int LDS_ELEMS = S * (WGX + WGY) * TK;
    static_assert(TK == 32 || TK == 64, "k-block");
    static_assert(FX * WX * 16 == WGX && FY * WY * 16 == WGY, "tile shape");
    // MFMA phase at raised wave priority: measured faster with 64-deep k-blocks (two-plane SYRK 2.65 -> 2.51
    // ms) and slower with 32-deep ones (three-plane SYRK 3.54 -> 3.91 ms)
    static constexpr bool PRIO = TK == 64;
};

__device__ inline f4 mfma(bf8 a, bf8 b, f4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }

// 16-byte load that keeps the pointer's address space (a global pointer stays a global load)
__device__ __forceinline__ u4 ld16(const __bf16* p) { return *(const u4*)p; }
__device__ __forceinline__ u4 ld16(const __attribute__((address_space(1))) __bf16* p) {
    return *(const __attribute__((address_space(1))) u4*)p;
}

// Operands lie in memory as fragments: 16 rows × 32 columns, the 64 lanes' 16-byte pieces in lane order
// (row r, columns 8g..8g+7 at piece 16g + r), 1 KB in a row.  A wave so moves a whole fragment with
// one load from a scalar address, coalesced: four neighbouring lanes read 64 bytes, where row-major
// operands give each lane of an MFMA operand its own row and the vector cache an access a lane (the two-
// plane half-transform below, nbf 768, 160 columns: 2.94 ms row-major, 2.16 by fragments).
constexpr int FRAG = 16 * KM;                                  // elements
__device__ __host__ inline size_t frag_elem(size_t row, size_t col, size_t ncol) {
    return ((row >> 4) * (ncol / KM) + col / KM) * FRAG + ((col % KM >> 3) * 16 + (row & 15)) * 8 + (col & 7);
}

__device__ const u4* pm_vec(const unsigned short*);   // the vector pointer of a mask pointer's address space
__device__ const __attribute__((address_space(1))) u4* pm_vec(const __attribute__((address_space(1))) unsigned short*);

__device__ u2* u2_ptr(__bf16*);
__device__ __attribute__((address_space(1))) u2* u2_ptr(__attribute__((address_space(1))) __bf16*);

// SYRK tile: D[ν][μ] over the np auxiliary columns of a split and ncol columns of M' each.
// Their fragment columns ("runs" of 32) follow each other and TK/32 make a k-block, so neither a
// column count nor a split has to fill whole k-blocks (past the last run: zeros).
// x / y: first fragment of the two operands' rows at the split's first auxiliary column and the
// spin's first column; row / pl / ps: elements between row fragments, planes and auxiliary
// columns; mask: the spin's sign masks (0x8000 flips), 16-byte aligned.  A wave that is not
// `live` only moves data.
// With SPLIT the leading product (plane 0 × plane 0) accumulates in acc and
// the correction products in acc2, so that FP32 rounding of the accumulators acts on the
// corrections at their own (2^-8 smaller) scale; the caller adds the two in FP64.
template <class C, bool SPLIT, class PX, class PM>
__device__ __forceinline__ void nt_tile2(__bf16* __restrict__ lds, PX x, PX y, size_t rowst, size_t pl, size_t ps,
                                         PM mask, int np, int ncol, bool live, f4 (&acc)[C::FX][C::FY],
                                         f4 (&acc2)[C::FX][C::FY]) {
    constexpr int S = C::S, NP = npairs<S>(), N = C::TK / KM, W = C::NT / 64;
    constexpr int RX = C::WGX / 16, RY = C::WGY / 16;            // row fragments of the tile
    constexpr int LX = RX * N / W, LY = RY * N / W;              // fragments a wave moves, a plane
    static_assert(W % N == 0 && LX * W == RX * N && LY * W == RY * N, "load shape");
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wx = wave % C::WX, wy = wave / C::WX;
    // this wave moves run `wave % N` of a k-block, row fragments wave/N, + W/N, ..
    const int slot = wave % N, rf0 = wave / N;
    auto Xs = [&](int k, int rf, int run) { return lds + ((k * (RX + RY) + rf) * N + run) * FRAG + lane * 8; };
    auto Ys = [&](int k, int rf, int run) { return Xs(k, RX + rf, run); };
#pragma unroll
    for (int i = 0; i < C::FX; ++i)
#pragma unroll
        for (int j = 0; j < C::FY; ++j) {
            acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};
            acc2[i][j] = f4{0.f, 0.f, 0.f, 0.f};
        }
    const int ncb = ncol / KM, nrun = np * ncb, nq = (nrun + N - 1) / N;
    if (nq <= 0) return;
    int run = slot, cb = slot % ncb;                             // of this wave's fragments, all uniform
    size_t off = (size_t)(slot / ncb) * ps + (size_t)cb * FRAG + rf0 * rowst;
    unsigned any = 0;                                            // a negative sign in this spin?
    for (int c = lane; c < ncol; c += 64) any |= mask[c];
    const bool neg = __any(any != 0);
    u4 rx[S][LX], ry[S][LY];
    int fcb = 0;                                                 // the fetched run's columns
    auto fetch = [&]() {
        fcb = cb;
        if (run < nrun) {
#pragma unroll
            for (int k = 0; k < S; ++k) {
#pragma unroll
                for (int j = 0; j < LX; ++j) rx[k][j] = ld16(x + off + k * pl + j * (W / N) * rowst + lane * 8);
#pragma unroll
                for (int j = 0; j < LY; ++j) ry[k][j] = ld16(y + off + k * pl + j * (W / N) * rowst + lane * 8);
            }
        } else {
#pragma unroll
            for (int k = 0; k < S; ++k) {
#pragma unroll
                for (int j = 0; j < LX; ++j) rx[k][j] = u4{0, 0, 0, 0};
#pragma unroll
                for (int j = 0; j < LY; ++j) ry[k][j] = u4{0, 0, 0, 0};
            }
        }
        run += N;
        cb += N;
        off += N * FRAG;
        while (cb >= ncb) {
            cb -= ncb;
            off += ps - (size_t)ncb * FRAG;
        }
    };
    auto stash = [&]() {
        if (neg) {
            const u4 rm = *(decltype(pm_vec(mask)))(mask + fcb * KM + (lane >> 4) * 8);
#pragma unroll
            for (int k = 0; k < S; ++k)
#pragma unroll
                for (int j = 0; j < LX; ++j) rx[k][j] ^= rm;
        }
#pragma unroll
        for (int k = 0; k < S; ++k) {
#pragma unroll
            for (int j = 0; j < LX; ++j) *(u4*)Xs(k, rf0 + j * (W / N), slot) = rx[k][j];
#pragma unroll
            for (int j = 0; j < LY; ++j) *(u4*)Ys(k, rf0 + j * (W / N), slot) = ry[k][j];
        }
    };
    auto compute = [&]() {
#pragma unroll
        for (int ks = 0; ks < N; ++ks) {
            bf8 fx[C::FX][S], fy[C::FY][S];
#pragma unroll
            for (int k = 0; k < S; ++k) {
#pragma unroll
                for (int i = 0; i < C::FX; ++i) fx[i][k] = *(const bf8*)Xs(k, wx * C::FX + i, ks);
#pragma unroll
                for (int j = 0; j < C::FY; ++j) fy[j][k] = *(const bf8*)Ys(k, wy * C::FY + j, ks);
            }
            // products outermost: consecutive MFMAs write different accumulators
#pragma unroll
            for (int p = 0; p < NP; ++p)
#pragma unroll
                for (int i = 0; i < C::FX; ++i)
#pragma unroll
                    for (int j = 0; j < C::FY; ++j) {
                        if (SPLIT && p > 0)
                            acc2[i][j] = mfma(fx[i][pa<S>(p)], fy[j][pb<S>(p)], acc2[i][j]);
                        else
                            acc[i][j] = mfma(fx[i][pa<S>(p)], fy[j][pb<S>(p)], acc[i][j]);
                    }
        }
    };
    // with C::PRIO the MFMA phase runs at raised wave priority, so that a wave ready to issue MFMAs
    // goes before the other waves' loads and LDS stashes (results unchanged)
    auto compute_prio = [&]() {
        if (!live) return;
        if constexpr (C::PRIO) __builtin_amdgcn_s_setprio(1);
        compute();
        if constexpr (C::PRIO) __builtin_amdgcn_s_setprio(0);
    };
    fetch();
    for (int q = 0; q < nq; ++q) {
        stash();
        __syncthreads();
        if (q + 1 < nq) fetch();
        compute_prio();
        __syncthreads();
    }
}

// One accumulator for every product.
template <class C, class PX, class PM>
__device__ __forceinline__ void nt_tile(__bf16* __restrict__ lds, PX x, PX y, size_t rowst, size_t pl, size_t ps, PM mask,
                                        int np, int ncol, bool live, f4 (&acc)[C::FX][C::FY]) {
    nt_tile2<C, false>(lds, x, y, rowst, pl, ps, mask, np, ncol, live, acc, acc);
}

// Planes of two values, packed (a in the low half).  One conversion instruction a plane; the empty asm keeps
// the compiler from joining the pairs into a wider vector conversion, which it can place in the
// registers of its own sources and order so that it overwrites them before they are read (clang of ROCm 7.2).
template <int S>
__device__ __forceinline__ void split_pair(float a, float b, unsigned (&w)[S]) {
#pragma unroll
    for (int k = 0; k < S; ++k) {
        w[k] = __builtin_bit_cast(unsigned, bf2{(__bf16)a, (__bf16)b});
        asm("" : "+v"(w[k]));
        a -= __builtin_bit_cast(float, w[k] << 16);
        b -= __builtin_bit_cast(float, w[k] & 0xffff0000u);
    }
}

// one accumulator fragment into the M' planes: lane holds columns c0 + 4(l/16) + r of row mu0 + l%16
template <int S, class P>
__device__ __forceinline__ void store_m(P m, size_t plane, int mu0, int c0, int nk, int lane, f4 a) {
    unsigned lo[S], hi[S];
    split_pair<S>(a[0], a[1], lo);
    split_pair<S>(a[2], a[3], hi);
    const size_t e = frag_elem(mu0, c0, nk) + (lane >> 5) * 128 + (lane & 15) * 8 + (lane >> 4 & 1) * 4;
#pragma unroll
    for (int k = 0; k < S; ++k) *(decltype(u2_ptr(m)))(m + k * plane + e) = u2{lo[k], hi[k]};
}

// ---------------------------------------------------------------------------
// Half-transform tile D[c][μ] = Σ_ν C'ᵀ[c][ν] Y[μ][ν]: 16·FX columns c by NW waves of 16·FM
// rows μ.  A wave's rows are its own, so its Y fragments go from memory straight into the
// registers the MFMA reads and only C'ᵀ, which all waves share, passes through LDS; with
// every column in one tile B is read once.  Y fragments of the next two steps of 32 ν are in
// flight while the MFMAs of this one run (each step reloads the registers it has consumed);
// C'ᵀ runs two steps ahead (one in registers, one in the other LDS buffer), one barrier
// a step.  Fragments of C'ᵀ beyond nk repeat the last one, and a wave with no row below nbf
// (`live` false) only stages.  Each sum runs over ν in steps of 32 with the plane products
// in order, whatever FX, FM and NW.  Bound by reading B's planes and writing M' where the columns
// are few: two planes, nbf 768, 160 columns, 3616 auxiliary: 3.14 ms before (64 × 256 tiles of both
// operands in LDS), 2.09 now = 4.9 TB/s and 980 TFLOP/s; three planes, nbf 645, 133 columns 4.00 -> 2.36 ms.
//
// Y: struct with  Raw  (what a fragment is loaded as), load(step, Raw (&)[FM]) and
// frag(const Raw&, bf8 (&)[S]).
template <int S_, int FX_, int FM_, int NW_>
struct HalfCfg {
    static constexpr int S = S_, FX = FX_, FM = FM_, NW = NW_, NT = NW * 64;
    static constexpr int TC = 16 * FX, TMU = 16 * FM * NW;      // tile columns and rows
    static constexpr int NX = (S * FX + NW - 1) / NW;           // fragments of C'ᵀ a wave moves in a step
    static constexpr int BUF = S * FX * FRAG;                   // elements of one LDS buffer
    static constexpr int LDS_ELEMS = 2 * BUF;
};

// ct: C'ᵀ fragments [S][nk/16][nu32], nu32 = padded ν / 32; c0 a multiple of 16
template <class H, bool SPLIT, class CT, class Y>
__device__ __forceinline__ void half_tile(__bf16* __restrict__ lds, CT ct, int nk, int nu32, int c0, int nst,
                                          bool live, Y& y, f4 (&acc)[H::FX][H::FM], f4 (&acc2)[H::FX][H::FM]) {
    constexpr int S = H::S, FX = H::FX, FM = H::FM, NP = npairs<S>();
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
    for (int i = 0; i < FX; ++i)
#pragma unroll
        for (int j = 0; j < FM; ++j) {
            acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};
            if constexpr (SPLIT) acc2[i][j] = f4{0.f, 0.f, 0.f, 0.f};
        }
    // this wave's fragments of a step: wave, wave + NW, .. of the S·FX (plane-major)
    const auto use = [&](int n) { return (n + 1) * H::NW <= S * FX || wave + n * H::NW < S * FX; };
    u4 rx[H::NX];
    auto xload = [&](int s) {
#pragma unroll
        for (int n = 0; n < H::NX; ++n)
            if (use(n)) {
                const int f = wave + n * H::NW, k = f / FX, row = min(c0 / 16 + f % FX, nk / 16 - 1);
                rx[n] = ld16(ct + ((size_t)(k * (nk / 16) + row) * nu32 + s) * FRAG + lane * 8);
            }
    };
    auto xstash = [&](auto b) {
#pragma unroll
        for (int n = 0; n < H::NX; ++n)
            if (use(n)) *(u4*)(lds + b() * H::BUF + (wave + n * H::NW) * FRAG + lane * 8) = rx[n];
    };
    typename Y::Raw ry[2][FM];
    auto compute = [&](auto b) {
        bf8 fy[FM][S];
#pragma unroll
        for (int j = 0; j < FM; ++j) y.frag(ry[b()][j], fy[j]);
#pragma unroll
        for (int i = 0; i < FX; ++i) {
            bf8 fx[S];
#pragma unroll
            for (int k = 0; k < S; ++k) fx[k] = *(const bf8*)(lds + b() * H::BUF + (k * FX + i) * FRAG + lane * 8);
#pragma unroll
            for (int p = 0; p < NP; ++p)
#pragma unroll
                for (int j = 0; j < FM; ++j) {
                    if (SPLIT && p > 0)
                        acc2[i][j] = mfma(fx[pa<S>(p)], fy[j][pb<S>(p)], acc2[i][j]);
                    else
                        acc[i][j] = mfma(fx[pa<S>(p)], fy[j][pb<S>(p)], acc[i][j]);
                }
        }
    };
    struct B0 { __device__ constexpr int operator()() const { return 0; } };
    struct B1 { __device__ constexpr int operator()() const { return 1; } };
    const int last = nst - 1;
    xload(0);
    if (live) {
        y.load(0, ry[0]);
        y.load(min(1, last), ry[1]);
    }
    xstash(B0{});
    xload(min(1, last));
    __syncthreads();
    // step s computes from buffer s % 2 while step s + 1's C'ᵀ goes into the other, last read at step
    // s - 1; steps past the last reload the last one, whose values nothing uses
    for (int s = 0;; s += 2) {
        xstash(B1{});
        xload(min(s + 2, last));
        if (live) {
            compute(B0{});
            y.load(min(s + 2, last), ry[0]);
        }
        if (s + 1 > last) break;
        __syncthreads();
        xstash(B0{});
        xload(min(s + 3, last));
        if (live) {
            compute(B1{});
            y.load(min(s + 3, last), ry[1]);
        }
        if (s + 2 > last) break;
        __syncthreads();
    }
}

}  // namespace bft
}  // namespace rjk
