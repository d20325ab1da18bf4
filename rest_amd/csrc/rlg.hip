// rlg.hip — the pair-block MLP of the learned initial guess: forward pass,
// masked-MSE loss, backward pass and Adam, all on the device (include/rest_lg.h).
//
// Activations, gradients and the master weights are FP32.  Every GEMM stages
// its operands in LDS as BF16 (round to nearest even) and multiplies them on
// the BF16 matrix cores (v_mfma_f32_16x16x32_bf16) with FP32 accumulation.
// Layout: row-major activations [batch][features], weights W_l [in][out]
// (Y = X W + b), SiLU after every hidden layer, linear output.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/rest_lg.h"

struct rlg_net {
    int device = 0;
    hipStream_t own = nullptr, stream = nullptr;
    std::vector<int> dims;   // n_in, hidden..., n_out
    size_t max_batch = 0, nparam = 0;
    float* params = nullptr;   // W_0, b_0, W_1, b_1, ... (FP32 master copy)
    float* grads = nullptr;    // same layout
    float* adam_m = nullptr;
    float* adam_v = nullptr;
    std::vector<size_t> w_off, b_off;
    std::vector<float*> act;   // act[0] = input copy pointer (not owned), act[l+1] = layer l output
    std::vector<float*> pre;   // pre-activation of every hidden layer
    float* g0 = nullptr;       // backward activation gradients (ping-pong)
    float* g1 = nullptr;
    float* split = nullptr;    // split-K partials of the weight gradients
    float* colsum = nullptr;   // their column sums of dZ (the bias gradients), one row a split
    size_t split_cap = 0;
    double* part = nullptr;    // loss partial sums
    long long step = 0;
    std::string err;
};

namespace {

typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int kTM = 64, kTN = 64, kTK = 64, kPad = 8;
constexpr int kLossBlocks = 512;

int fail(rlg_net* n, int code, const std::string& m) {
    if (n) n->err = m;
    return code;
}

#define RLG_HIP(net, call)                                                                              \
    do {                                                                                                \
        hipError_t e_ = (call);                                                                         \
        if (e_ != hipSuccess) return fail((net), RLG_ERR_HIP, std::string(#call) + ": " + hipGetErrorString(e_)); \
    } while (0)

__device__ inline float sigmoid(float z) { return 1.f / (1.f + __expf(-z)); }

// What the GEMM does with C(m, n) = Σ_k A(m,k) B(k,n) before it leaves the registers
enum { EPI_NONE, EPI_SILU, EPI_LINEAR, EPI_SILU_BWD };
struct Epi {
    const float* bias = nullptr;   // SILU, LINEAR: per column n
    float* act = nullptr;          // SILU: C = z = sum + bias, act = SiLU(z)
    const float* pre = nullptr;    // SILU_BWD: C = sum · SiLU'(pre)
    float* colsum = nullptr;       // NONE: Σ_k B(k,n) of split z in FP32 at colsum + z·N (the bias gradient)
};

// C_z[m][n] = Σ_{k in split z} A(m,k) B(k,n),  A(m,k) = A[m*sam + k*sak], B(k,n) = B[k*sbk + n*sbn];
// split z covers k in [z*kchunk, min(K, (z+1)*kchunk)) and writes C + z*M*ldc.
// AK / BK: neighbouring threads of a load take neighbouring k (else neighbouring m / n); the launcher
// picks the one that is contiguous in memory.  The network's products are short (K 196..512 a split) and
// bound by the latency of their loads: the next 64-deep block is fetched while the current one is
// multiplied, and bias, SiLU, SiLU' and the column sums ride along.  Batch 4096 of the packaged network: a
// product 45 -> 12-16 us, loss and gradient 4.39 -> 0.29 ms (17 launches, and the copy to the host).
// Sums run over k in ascending blocks of 32 whatever the block depth.
template <bool AK, bool BK, int EPI>
__global__ __launch_bounds__(256) void k_gemm(const float* __restrict__ A, long sam, long sak,
                                              const float* __restrict__ B, long sbk, long sbn,
                                              float* __restrict__ C, long ldc, int M, int N, int K, int kchunk, Epi ep) {
    constexpr int NL = kTM * kTK / 256;      // elements a thread loads of either operand
    static_assert(kTM == kTN, "both operands load alike");
    __shared__ __align__(16) __bf16 As[kTM][kTK + kPad];
    __shared__ __align__(16) __bf16 Bt[kTN][kTK + kPad];   // B tile stored transposed: Bt[n][k]
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int m0 = blockIdx.y * kTM, n0 = blockIdx.x * kTN;
    const int kbeg = blockIdx.z * kchunk, kend = min(K, kbeg + kchunk);
    C += (size_t)blockIdx.z * M * ldc;
    const int wm = w >> 1, wn = w & 1;
    const bool sums = EPI == EPI_NONE && ep.colsum && blockIdx.y == 0;
    float ra[NL], rb[NL], cs = 0.f;
    // element i of a thread: (row, k) of the 64 × kTK tile
    auto at = [&](bool kfast, int i, int* r, int* kk) {
        if (kfast) {
            *kk = tid % kTK;
            *r = tid / kTK + i * (256 / kTK);
        } else {
            *r = tid % kTM;
            *kk = tid / kTM + i * (256 / kTM);
        }
    };
    auto fetch = [&](int k0) {
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            int r, kk;
            at(AK, i, &r, &kk);
            const bool in = m0 + r < M && k0 + kk < kend;
            ra[i] = in ? A[(size_t)(m0 + r) * sam + (size_t)(k0 + kk) * sak] : 0.f;
        }
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            int r, kk;
            at(BK, i, &r, &kk);
            const bool in = n0 + r < N && k0 + kk < kend;
            rb[i] = in ? B[(size_t)(k0 + kk) * sbk + (size_t)(n0 + r) * sbn] : 0.f;
        }
    };
    f4 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};
    if (kbeg < kend) fetch(kbeg);
    for (int k0 = kbeg; k0 < kend; k0 += kTK) {
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            int r, kk;
            at(AK, i, &r, &kk);
            As[r][kk] = (__bf16)ra[i];
            at(BK, i, &r, &kk);
            Bt[r][kk] = (__bf16)rb[i];
            if (sums && !BK) cs += rb[i];
        }
        __syncthreads();
        if (k0 + kTK < kend) fetch(k0 + kTK);
#pragma unroll
        for (int ks = 0; ks < kTK; ks += 32) {
            bf8 a[2], b[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) a[i] = *(const bf8*)&As[wm * 32 + i * 16 + (lane & 15)][ks + 8 * (lane >> 4)];
#pragma unroll
            for (int j = 0; j < 2; ++j) b[j] = *(const bf8*)&Bt[wn * 32 + j * 16 + (lane & 15)][ks + 8 * (lane >> 4)];
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
        }
        __syncthreads();
    }
    // D[4(l/16)+r][l%16] of each 16x16 block
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int gm = m0 + wm * 32 + i * 16 + 4 * (lane >> 4) + r;
                const int gn = n0 + wn * 32 + j * 16 + (lane & 15);
                if (gm >= M || gn >= N) continue;
                const size_t o = (size_t)gm * ldc + gn;
                float v = acc[i][j][r];
                if (EPI == EPI_SILU || EPI == EPI_LINEAR) v += ep.bias[gn];
                if (EPI == EPI_SILU) ep.act[o] = v * sigmoid(v);
                if (EPI == EPI_SILU_BWD) {
                    const float z = ep.pre[o], s = sigmoid(z);
                    v = v * s * (1.f + z * (1.f - s));
                }
                C[o] = v;
            }
    if (sums && !BK) {   // column tid % 64 is spread over four threads
        float* red = (float*)&As[0][0];
        red[tid] = cs;
        __syncthreads();
        if (tid < kTN && n0 + tid < N)
            ep.colsum[(size_t)blockIdx.z * N + n0 + tid] = (red[tid] + red[tid + 64]) + (red[tid + 128] + red[tid + 192]);
    }
}

// partial[2b] = Σ mask·(y − t)², partial[2b+1] = Σ mask   (FP64 sums)
__global__ void k_loss_sums(const float* __restrict__ Y, const float* __restrict__ T, const float* __restrict__ Mk,
                            size_t n, double* __restrict__ partial) {
    __shared__ double s0[256], s1[256];
    double a = 0.0, c = 0.0;
    for (size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (size_t)gridDim.x * blockDim.x) {
        const double d = (double)Y[t] - (double)T[t];
        a += (double)Mk[t] * d * d;
        c += (double)Mk[t];
    }
    s0[threadIdx.x] = a;
    s1[threadIdx.x] = c;
    __syncthreads();
    for (int off = 128; off > 0; off >>= 1) {
        if ((int)threadIdx.x < off) {
            s0[threadIdx.x] += s0[threadIdx.x + off];
            s1[threadIdx.x] += s1[threadIdx.x + off];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        partial[2 * blockIdx.x] = s0[0];
        partial[2 * blockIdx.x + 1] = s1[0];
    }
}

// G = 2 mask (y − t) / Σmask
__global__ void k_loss_grad(const float* __restrict__ Y, const float* __restrict__ T, const float* __restrict__ Mk,
                            size_t n, float scale, float* __restrict__ G) {
    for (size_t t = (size_t)blockIdx.x * 256 + threadIdx.x; t < n; t += (size_t)gridDim.x * 256)
        G[t] = scale * Mk[t] * (Y[t] - T[t]);
}

// out[i] = Σ_z part[z*count + i] for the weight gradient (i < count), then the bias gradient from
// colsum[z*nb + i] (nb columns).  The bias gradient used to be one thread a column over the whole
// batch: 937 of 1085 us a layer at batch 4096.
__global__ void k_sum_splits(const float* __restrict__ part, const float* __restrict__ colsum, int splits, size_t count,
                             int nb, float* __restrict__ out) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= count + nb) return;
    const float* src = t < count ? part + t : colsum + (t - count);
    const size_t step = t < count ? count : (size_t)nb;
    float s = 0.f;
    for (int z = 0; z < splits; ++z) s += src[(size_t)z * step];
    out[t] = s;
}

__global__ void k_adam(float* __restrict__ w, const float* __restrict__ g, float* __restrict__ m,
                       float* __restrict__ v, size_t n, float lr, float b1, float b2, float eps, float bc1,
                       float bc2) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const float gi = g[t];
    const float mi = b1 * m[t] + (1.f - b1) * gi;
    const float vi = b2 * v[t] + (1.f - b2) * gi * gi;
    m[t] = mi;
    v[t] = vi;
    w[t] -= lr * (mi / bc1) / (sqrtf(vi / bc2) + eps);
}

unsigned blocks(size_t n, unsigned b = 256) { return (unsigned)((n + b - 1) / b); }

template <int EPI>
hipError_t gemm_t(hipStream_t st, const float* A, long sam, long sak, const float* B, long sbk, long sbn, float* C,
                  long ldc, int M, int N, int K, int splits, const Epi& ep) {
    const int kchunk = ((K + splits - 1) / splits + 31) / 32 * 32;
    dim3 grid(blocks(N, kTN), blocks(M, kTM), splits);
    auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, grid, dim3(256), 0, st, A, sam, sak, B, sbk, sbn, C, ldc, M, N, K, kchunk, ep);
        return hipGetLastError();
    };
    const bool bk = sbk == 1 && sbn != 1;   // a one-column B keeps the path that forms column sums
    if constexpr (EPI == EPI_SILU || EPI == EPI_LINEAR) return go(k_gemm<true, false, EPI>);   // forward: A's rows, W's rows
    if constexpr (EPI == EPI_SILU_BWD) return bk ? go(k_gemm<true, true, EPI>) : go(k_gemm<true, false, EPI>);
    if (sak == 1) return bk ? go(k_gemm<true, true, EPI>) : go(k_gemm<true, false, EPI>);
    return bk ? go(k_gemm<false, true, EPI>) : go(k_gemm<false, false, EPI>);
}

hipError_t gemm(hipStream_t st, const float* A, long sam, long sak, const float* B, long sbk, long sbn, float* C,
                long ldc, int M, int N, int K, int splits) {
    return gemm_t<EPI_NONE>(st, A, sam, sak, B, sbk, sbn, C, ldc, M, N, K, splits, Epi());
}

int nlayers(const rlg_net* n) { return (int)n->dims.size() - 1; }

// forward over `batch` rows of x; the last layer's output goes to y (batch × n_out)
int forward(rlg_net* n, const float* x, size_t batch, float* y) {
    const int L = nlayers(n);
    n->act[0] = const_cast<float*>(x);
    for (int l = 0; l < L; ++l) {
        const int din = n->dims[l], dout = n->dims[l + 1];
        Epi ep;
        ep.bias = n->params + n->b_off[l];
        ep.act = n->act[l + 1];
        if (l + 1 < L)
            RLG_HIP(n, gemm_t<EPI_SILU>(n->stream, n->act[l], din, 1, n->params + n->w_off[l], dout, 1, n->pre[l], dout,
                                        (int)batch, dout, din, 1, ep));
        else
            RLG_HIP(n, gemm_t<EPI_LINEAR>(n->stream, n->act[l], din, 1, n->params + n->w_off[l], dout, 1, y, dout,
                                          (int)batch, dout, din, 1, ep));
    }
    return RLG_OK;
}

int check_batch(rlg_net* n, size_t batch) {
    if (batch == 0 || batch > n->max_batch)
        return fail(n, RLG_ERR_ARG, "batch must be 1.." + std::to_string(n->max_batch));
    return RLG_OK;
}

}  // namespace

extern "C" {

int rlg_create(int device, size_t n_in, size_t n_hidden, size_t n_hidden_layers, size_t n_out, size_t max_batch,
               rlg_net** out) {
    if (!out || n_in == 0 || n_hidden == 0 || n_out == 0 || max_batch == 0 || n_hidden_layers > 16 ||
        n_in > 65536 || n_hidden > 65536 || n_out > 65536 || max_batch > (size_t(1) << 24))
        return RLG_ERR_ARG;
    *out = nullptr;
    rlg_net* n = new rlg_net();
    n->device = device;
    n->dims.push_back((int)n_in);
    for (size_t i = 0; i < n_hidden_layers; ++i) n->dims.push_back((int)n_hidden);
    n->dims.push_back((int)n_out);
    n->max_batch = max_batch;
    const int L = nlayers(n);
    size_t off = 0, widest = 0;
    for (int l = 0; l < L; ++l) {
        n->w_off.push_back(off);
        off += (size_t)n->dims[l] * n->dims[l + 1];
        n->b_off.push_back(off);
        off += n->dims[l + 1];
        widest = std::max(widest, (size_t)std::max(n->dims[l], n->dims[l + 1]));
    }
    n->nparam = off;
    auto alloc = [&](float** p, size_t cnt) { return hipMalloc((void**)p, cnt * sizeof(float)) == hipSuccess; };
    bool ok = hipSetDevice(device) == hipSuccess && hipStreamCreate(&n->own) == hipSuccess;
    n->stream = n->own;
    ok = ok && alloc(&n->params, off) && alloc(&n->grads, off) && alloc(&n->adam_m, off) && alloc(&n->adam_v, off);
    n->act.assign(L + 1, nullptr);
    n->pre.assign(L - 1, nullptr);
    for (int l = 0; l < L && ok; ++l) {
        ok = alloc(&n->act[l + 1], max_batch * n->dims[l + 1]);
        if (l + 1 < L) ok = ok && alloc(&n->pre[l], max_batch * n->dims[l + 1]);
    }
    ok = ok && alloc(&n->g0, max_batch * widest) && alloc(&n->g1, max_batch * widest);
    ok = ok && hipMalloc((void**)&n->part, 2 * kLossBlocks * sizeof(double)) == hipSuccess;
    // split-K partials for the largest weight gradient
    size_t wmax = 0;
    for (int l = 0; l < L; ++l) wmax = std::max(wmax, (size_t)n->dims[l] * n->dims[l + 1]);
    n->split_cap = 16 * wmax;
    ok = ok && alloc(&n->split, n->split_cap) && alloc(&n->colsum, 16 * widest);
    ok = ok && hipMemsetAsync(n->params, 0, off * sizeof(float), n->stream) == hipSuccess &&
         hipMemsetAsync(n->adam_m, 0, off * sizeof(float), n->stream) == hipSuccess &&
         hipMemsetAsync(n->adam_v, 0, off * sizeof(float), n->stream) == hipSuccess &&
         hipStreamSynchronize(n->stream) == hipSuccess;
    if (!ok) {
        rlg_destroy(n);
        return RLG_ERR_NOMEM;
    }
    *out = n;
    return RLG_OK;
}

int rlg_destroy(rlg_net* n) {
    if (!n) return RLG_OK;
    (void)hipSetDevice(n->device);
    if (n->stream) (void)hipStreamSynchronize(n->stream);
    for (float* p : {n->params, n->grads, n->adam_m, n->adam_v, n->g0, n->g1, n->split, n->colsum})
        if (p) (void)hipFree(p);
    for (float* p : n->pre)
        if (p) (void)hipFree(p);
    for (size_t l = 1; l < n->act.size(); ++l)
        if (n->act[l]) (void)hipFree(n->act[l]);
    if (n->part) (void)hipFree(n->part);
    if (n->own) (void)hipStreamDestroy(n->own);
    delete n;
    return RLG_OK;
}

const char* rlg_last_error(const rlg_net* n) { return n ? n->err.c_str() : "NULL network"; }

size_t rlg_num_params(const rlg_net* n) { return n ? n->nparam : 0; }

int rlg_set_stream(rlg_net* n, void* stream) {
    if (!n) return RLG_ERR_ARG;
    n->stream = stream ? (hipStream_t)stream : n->own;
    return RLG_OK;
}

int rlg_set_params(rlg_net* n, const float* host) {
    if (!n || !host) return RLG_ERR_ARG;
    RLG_HIP(n, hipSetDevice(n->device));
    RLG_HIP(n, hipMemcpyAsync(n->params, host, n->nparam * sizeof(float), hipMemcpyHostToDevice, n->stream));
    RLG_HIP(n, hipStreamSynchronize(n->stream));
    return RLG_OK;
}

int rlg_get_params(rlg_net* n, float* host) {
    if (!n || !host) return RLG_ERR_ARG;
    RLG_HIP(n, hipSetDevice(n->device));
    RLG_HIP(n, hipMemcpyAsync(host, n->params, n->nparam * sizeof(float), hipMemcpyDeviceToHost, n->stream));
    RLG_HIP(n, hipStreamSynchronize(n->stream));
    return RLG_OK;
}

int rlg_forward(rlg_net* n, const float* x_dev, size_t batch, float* y_dev) {
    if (!n || !x_dev || !y_dev) return fail(n, RLG_ERR_ARG, "rlg_forward: NULL argument");
    int rc = check_batch(n, batch);
    if (rc) return rc;
    RLG_HIP(n, hipSetDevice(n->device));
    // without a hidden layer the one product reads x_dev while it writes: overlapping arrays take the copy
    const size_t nx = batch * n->dims.front(), ny = batch * n->dims.back();
    const bool overlap = nlayers(n) == 1 && (uintptr_t)x_dev < (uintptr_t)(y_dev + ny) && (uintptr_t)y_dev < (uintptr_t)(x_dev + nx);
    float* const y = overlap ? n->act.back() : y_dev;
    rc = forward(n, x_dev, batch, y);
    if (rc) return rc;
    if (overlap)
        RLG_HIP(n, hipMemcpyAsync(y_dev, y, ny * sizeof(float), hipMemcpyDeviceToDevice, n->stream));
    RLG_HIP(n, hipStreamSynchronize(n->stream));
    return RLG_OK;
}

int rlg_loss_grad(rlg_net* n, const float* x_dev, const float* t_dev, const float* mask_dev, size_t batch,
                  double* loss, float* grad_host) {
    if (!n || !x_dev || !t_dev || !mask_dev) return fail(n, RLG_ERR_ARG, "rlg_loss_grad: NULL argument");
    int rc = check_batch(n, batch);
    if (rc) return rc;
    RLG_HIP(n, hipSetDevice(n->device));
    float* y = n->act.back();
    rc = forward(n, x_dev, batch, y);
    if (rc) return rc;
    const int L = nlayers(n), nout = n->dims.back();
    const size_t ny = batch * nout;
    hipLaunchKernelGGL(k_loss_sums, dim3(kLossBlocks), dim3(256), 0, n->stream, y, t_dev, mask_dev, ny, n->part);
    RLG_HIP(n, hipGetLastError());
    std::vector<double> part(2 * kLossBlocks);
    RLG_HIP(n, hipMemcpyAsync(part.data(), n->part, part.size() * sizeof(double), hipMemcpyDeviceToHost, n->stream));
    RLG_HIP(n, hipStreamSynchronize(n->stream));
    double se = 0.0, msum = 0.0;
    for (int b = 0; b < kLossBlocks; ++b) {
        se += part[2 * b];
        msum += part[2 * b + 1];
    }
    if (!(msum > 0.0)) return fail(n, RLG_ERR_ARG, "rlg_loss_grad: the mask is empty");
    if (loss) *loss = se / msum;
    float* G = n->g0;
    float* Gn = n->g1;
    hipLaunchKernelGGL(k_loss_grad, dim3(std::min(blocks(ny), 1024u)), dim3(256), 0, n->stream, y, t_dev, mask_dev, ny,
                       (float)(2.0 / msum), G);
    RLG_HIP(n, hipGetLastError());
    for (int l = L - 1; l >= 0; --l) {
        const int din = n->dims[l], dout = n->dims[l + 1];
        float* dZ = G;
        // gW = A_lᵀ dZ  (din × dout, reduction over the batch, split over rows of the batch), and the
        // column sums of dZ for the bias in the same pass
        const size_t wcount = (size_t)din * dout;
        int splits = (int)std::min<size_t>(16, std::max<size_t>(1, batch / 256));
        splits = (int)std::min<size_t>(splits, n->split_cap / wcount);
        Epi ep;
        ep.colsum = n->colsum;
        RLG_HIP(n, gemm_t<EPI_NONE>(n->stream, n->act[l], 1, din, dZ, dout, 1, n->split, dout, din, dout, (int)batch,
                                    splits, ep));
        hipLaunchKernelGGL(k_sum_splits, dim3(blocks(wcount + dout)), dim3(256), 0, n->stream, n->split, n->colsum,
                           splits, wcount, dout, n->grads + n->w_off[l]);   // the bias follows its weights
        RLG_HIP(n, hipGetLastError());
        if (l > 0) {   // dZ_{l-1} = (dZ W_lᵀ) ⊙ SiLU'(pre_{l-1})  (batch × din)
            Epi eb;
            eb.pre = n->pre[l - 1];
            RLG_HIP(n, gemm_t<EPI_SILU_BWD>(n->stream, dZ, dout, 1, n->params + n->w_off[l], 1, dout, Gn, din,
                                            (int)batch, din, dout, 1, eb));
            std::swap(G, Gn);
        }
    }
    if (grad_host)
        RLG_HIP(n, hipMemcpyAsync(grad_host, n->grads, n->nparam * sizeof(float), hipMemcpyDeviceToHost, n->stream));
    RLG_HIP(n, hipStreamSynchronize(n->stream));
    return RLG_OK;
}

int rlg_adam_step(rlg_net* n, double lr, double beta1, double beta2, double eps) {
    if (!n) return RLG_ERR_ARG;
    if (!(lr > 0) || !(beta1 >= 0 && beta1 < 1) || !(beta2 >= 0 && beta2 < 1) || !(eps > 0))
        return fail(n, RLG_ERR_ARG, "rlg_adam_step: need lr > 0, 0 <= beta < 1, eps > 0");
    RLG_HIP(n, hipSetDevice(n->device));
    ++n->step;
    const float bc1 = (float)(1.0 - std::pow(beta1, (double)n->step));
    const float bc2 = (float)(1.0 - std::pow(beta2, (double)n->step));
    hipLaunchKernelGGL(k_adam, dim3(blocks(n->nparam)), dim3(256), 0, n->stream, n->params, n->grads, n->adam_m,
                       n->adam_v, n->nparam, (float)lr, (float)beta1, (float)beta2, (float)eps, bc1, bc2);
    RLG_HIP(n, hipGetLastError());
    RLG_HIP(n, hipStreamSynchronize(n->stream));
    return RLG_OK;
}

int rlg_reset_optimizer(rlg_net* n) {
    if (!n) return RLG_ERR_ARG;
    RLG_HIP(n, hipSetDevice(n->device));
    RLG_HIP(n, hipMemsetAsync(n->adam_m, 0, n->nparam * sizeof(float), n->stream));
    RLG_HIP(n, hipMemsetAsync(n->adam_v, 0, n->nparam * sizeof(float), n->stream));
    RLG_HIP(n, hipStreamSynchronize(n->stream));
    n->step = 0;
    return RLG_OK;
}

int rlg_gemm_bf16(rlg_net* n, const float* A, long sam, long sak, const float* B, long sbk, long sbn, float* C,
                  long ldc, int M, int N, int K) {
    if (!n || !A || !B || !C || M <= 0 || N <= 0 || K <= 0 || ldc < N)
        return fail(n, RLG_ERR_ARG, "rlg_gemm_bf16: bad argument");
    RLG_HIP(n, hipSetDevice(n->device));
    RLG_HIP(n, gemm(n->stream, A, sam, sak, B, sbk, sbn, C, ldc, M, N, K, 1));
    RLG_HIP(n, hipStreamSynchronize(n->stream));
    return RLG_OK;
}

}  // extern "C"
