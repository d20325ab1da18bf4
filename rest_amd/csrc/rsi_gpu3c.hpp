// rsi_gpu3c.hpp — device three-centre integrals (μν|P) for the B producer.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <vector>

#include "rsi_internal.hpp"

namespace rsi {

// A shell as the device kernels read it; primitives and the Cartesian ->
// spherical rows live in flat arrays at p0 / t0.
struct GShell {
    double A[3];
    int l, nprim, p0, t0, off, pad;
};

constexpr int kGpuMaxLOrb = 2;   // orbital shells up to d
constexpr int kGpuMaxLAux = 4;   // auxiliary shells up to g
constexpr int kGpuClasses = (kGpuMaxLOrb + 1) * (kGpuMaxLOrb + 2) / 2;   // (la >= lb) pairs

// A shell pair (or, for the metric, one auxiliary shell a): its primitive pairs are k0 .. k0 + nk of the
// slab's list, their Hermite coefficients start at e0.
struct GPair {
    int a, b, k0, nk;
    size_t e0;
};
struct GPrim {
    int pair, ia, ib, k;   // primitive pair k of its pair (index into the whole pair list)
};

struct Gpu3c {
    void* arena = nullptr;    // the one allocation that holds all of the following
    GShell* orb = nullptr;
    GShell* aux = nullptr;
    double* pexp = nullptr;
    double* pcoef = nullptr;
    double* tsph = nullptr;
    double* boys = nullptr;   // Boys table, rows of Boys::kMTab at T = i·Boys::kStep
    int* auxl = nullptr;      // auxiliary shells grouped by l
    GPair* pairs = nullptr;   // screened shell pairs (A.l >= B.l), grouped by slab, then class
    GPrim* prims = nullptr;   // their primitive pairs above the cut-off, in the same order
    GPair* mpairs = nullptr;  // auxiliary shells as the metric's pairs, grouped by l
    GPrim* mprims = nullptr;
    double* pp = nullptr;     // (p, P) of the current slab's primitive pairs
    double* E = nullptr;      // their Hermite coefficients
    int aux_off[kGpuMaxLAux + 1] = {}, aux_cnt[kGpuMaxLAux + 1] = {};
    int mprim_off[kGpuMaxLAux + 1] = {}, mprim_cnt[kGpuMaxLAux + 1] = {};
    std::vector<size_t> cuts;   // slab boundaries in pair columns j
    std::vector<size_t> cls_off, cls_cnt, prim_off, prim_cnt;   // [slab * kGpuClasses + class]
    std::vector<size_t> dropped;                                // pairs of a slab that screening removed
};

bool gpu3c_supported(const Basis& orb, const Basis& aux);
bool gpu3c_aux_supported(const Basis& aux);
// Upload shells, primitives, transforms and the Boys table; build the pair lists of every slab
// [cuts[k], cuts[k+1]) (orb may be null with no cuts: the metric alone).  Returns an RJK_* code.
int gpu3c_init(Gpu3c* g, const Basis* orb, const Basis& aux, const std::vector<size_t>& cuts, hipStream_t st);
// (μν|P) of slab k into the device array X[naux][nq] (every element is written), on st.
int gpu3c_slab(const Gpu3c& g, size_t k, hipStream_t st, double* X, size_t naux);
// the metric (P|Q), both triangles, into the device array V[naux][naux], on st
int gpu2c(const Gpu3c& g, hipStream_t st, double* V, size_t naux);
void gpu3c_free(Gpu3c* g);

}  // namespace rsi
