// mlp.hip -- the learned step-size proposer: a 12 -> 64 -> 64 -> 1 MLP with
// tanh hidden layers, BF16 weights (FP32 master copies for Adam) and FP32
// accumulation.  Forward, backward (per-block gradient partials reduced in a
// fixed order, so gradients are deterministic) and Adam run on the GPU.
//
// Parameter vector layout (FP32 master / BF16 working copy), kNParam floats:
//   W1[12][64] | b1[64] | W2[64][64] | b2[64] | w3[64] | b3
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <random>
#include <string>
#include <vector>

#include "../../include/red_abi.h"
#include "device_scope.hpp"
#include "mlp.hpp"

namespace rdamd {

constexpr int kIn = RD_MLP_IN, kH = RD_MLP_HIDDEN;
constexpr int kOffW1 = 0, kOffB1 = kIn * kH, kOffW2 = kOffB1 + kH, kOffB2 = kOffW2 + kH * kH, kOffW3 = kOffB2 + kH,
              kOffB3 = kOffW3 + kH;
constexpr int kNParam = kOffB3 + 1;
static_assert(kNParam == RD_MLP_NPARAM, "parameter count");
constexpr int kGradBlock = 256;   // threads of a gradient block
constexpr int kGradRows = 64;     // its samples

__device__ inline float bf16_to_f32(uint16_t h)
{
    return __uint_as_float((uint32_t)h << 16);
}
__host__ __device__ inline uint16_t f32_to_bf16(float f)
{
    // round to nearest even
    uint32_t u;
    std::memcpy(&u, &f, 4);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);   // NaN
    const uint32_t r = ((u >> 16) & 1u) + 0x7fffu;
    return (uint16_t)((u + r) >> 16);
}

// Standardisation and target.  The network's output y' is de-normalised to
// y' t_std + t_mean + x[base] (base < 0: no offset), so a network trained on
// targets t - x[base] still returns log h.  quantile 0 trains the mean
// (loss 0.5 e^2); quantile q in (0, 1) trains the q-quantile (pinball loss
// max(q u, (q - 1) u), u = t' - y').
struct Norm {
    float mean[kIn], inv_std[kIn];
    float t_mean, t_std;
    int base;
    float quantile;
};

// Inference: raw features -> log h (de-normalised).  One wave per sample,
// lane j = hidden unit j: layer 1 and layer 2 are 12- and 64-term dot
// products per lane over inputs held in LDS; the output sums the 64 lanes'
// w3_j h2_j with a fixed butterfly, so results are reproducible.
__global__ __launch_bounds__(kH) void k_mlp_forward(const uint16_t* __restrict__ wb, Norm nm,
                                                    const float* __restrict__ xraw, uint32_t n,
                                                    float* __restrict__ y)
{
    static_assert(kH == 64, "one lane per hidden unit of a 64-wide wave");
    __shared__ float xs[kIn];
    __shared__ float h1[kH];
    const uint32_t q = blockIdx.x;
    const uint32_t j = threadIdx.x;
    if (q >= n) return;
    if (j < (uint32_t)kIn) xs[j] = (xraw[(size_t)q * kIn + j] - nm.mean[j]) * nm.inv_std[j];
    __syncthreads();
    float a = bf16_to_f32(wb[kOffB1 + j]);
#pragma unroll
    for (int i = 0; i < kIn; ++i) a = fmaf(xs[i], bf16_to_f32(wb[kOffW1 + i * kH + j]), a);
    h1[j] = tanhf(a);
    __syncthreads();
    float b = bf16_to_f32(wb[kOffB2 + j]);
#pragma unroll 16
    for (int k = 0; k < kH; ++k) b = fmaf(h1[k], bf16_to_f32(wb[kOffW2 + k * kH + j]), b);
    float o = tanhf(b) * bf16_to_f32(wb[kOffW3 + j]);
    for (int off = 32; off > 0; off >>= 1) o += __shfl_xor(o, off, 64);
    if (j == 0) {
        const float off = nm.base >= 0 ? xraw[(size_t)q * kIn + nm.base] : 0.0f;
        y[q] = (o + bf16_to_f32(wb[kOffB3])) * nm.t_std + nm.t_mean + off;
    }
}

typedef float f32x4 __attribute__((ext_vector_type(4)));

// D += A B for a 16 x 16 tile over 4 terms, in FP32 (v_mfma_f32_16x16x4_f32).
// Lane l holds A[l % 16][l / 16], B[l / 16][l % 16] and D[4 (l / 16) + r][l % 16],
// r = 0..3.
__device__ inline f32x4 mfma4(float a, float b, f32x4 d) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, d, 0, 0, 0); }

// Loss in normalised target units -- 0.5 mean e^2, or the mean pinball loss
// when nm.quantile > 0 (e = y' - t') -- and its gradient.
// A block of four waves takes 64 samples: wave w their rows 16 w .. 16 w + 15
// through both layers and back, and rows or columns 16 w .. of every sum over the
// samples, all of them 16 x 16 tiles of FP32 matrix instructions on operands
// in LDS (a plain sum is a product with ones).  Weights are BF16 values held in
// FP32; each result is one chain of fused multiply-adds in ascending order
// from its bias or zero, so it has the bits of the scalar loop over the same
// terms.  Each block leaves its partial gradient (and loss) in part[block][*];
// k_mlp_reduce sums them in block order.
// Bound by the matrix instructions (about 1000 per block, 33 cycles each on one
// of four SIMDs) and 8192 tanh.  (One sample per lane of a single wave, its
// activations in scratch, took 110 us for 20000 samples, this 28.)
constexpr int kLd = kH + 4;   // LDS row length: rows 4 banks apart, so 16 rows x 4 columns touch every bank once
__global__ __launch_bounds__(kGradBlock) void k_mlp_grad(const uint16_t* __restrict__ wb, Norm nm,
                                                         const float* __restrict__ xraw,
                                                         const float* __restrict__ tr,
                                                         const uint32_t* __restrict__ idx, uint32_t n, float scale,
                                                         float* __restrict__ part)
{
    static_assert(kH == 64 && kIn <= 16 && kGradBlock == 256 && kGradRows == 64, "tile shape");
    __shared__ float W1[12][kLd], W2[kH][kLd], w3[kH], b1[kH], b2[kH];
    __shared__ float X[kGradRows][20], A[kGradRows][kLd], B[kGradRows][kLd], H[kGradRows][kLd];
    __shared__ float st[kGradRows], sdy[kGradRows], sloss[kGradRows];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int lc = lane & 15, lr = lane >> 4;
    const int row0 = 16 * w;
    const uint32_t q0 = blockIdx.x * kGradRows;
    for (int k = tid; k < kIn * kH; k += kGradBlock) W1[k / kH][k % kH] = bf16_to_f32(wb[kOffW1 + k]);
    for (int k = tid; k < kH * kH; k += kGradBlock) W2[k / kH][k % kH] = bf16_to_f32(wb[kOffW2 + k]);
    if (tid < kH) {
        w3[tid] = bf16_to_f32(wb[kOffW3 + tid]);
        b1[tid] = bf16_to_f32(wb[kOffB1 + tid]);
        b2[tid] = bf16_to_f32(wb[kOffB2 + tid]);
    }
    const float b3 = bf16_to_f32(wb[kOffB3]);
    // normalised inputs (columns kIn..15 and rows past the end: 0) and targets
    for (int k = tid; k < kGradRows * 16; k += kGradBlock) {
        const int r = k / 16, c = k % 16;
        float v = 0.0f;
        if (q0 + r < n && c < kIn) {
            const uint32_t src = idx ? idx[q0 + r] : q0 + r;
            v = (xraw[(size_t)src * kIn + c] - nm.mean[c]) * nm.inv_std[c];
        }
        X[r][c] = v;
    }
    if (tid < kGradRows) {
        float v = 0.0f;
        if (q0 + tid < n) {
            const uint32_t src = idx ? idx[q0 + tid] : q0 + tid;
            const float tb = tr[src] - (nm.base >= 0 ? xraw[(size_t)src * kIn + nm.base] : 0.0f);
            v = (tb - nm.t_mean) / nm.t_std;
        }
        st[tid] = v;
    }
    __syncthreads();
    bool in[4];   // this lane's rows of a tile: row0 + 4 lr + r
#pragma unroll
    for (int r = 0; r < 4; ++r) in[r] = q0 + row0 + 4 * lr + r < n;
    // layer 1: h1 = tanh(b1 + X W1), rows of this wave; rows past the end: 0
    f32x4 h1[4], h2[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const float b = b1[16 * c + lc];
        h1[c] = f32x4{b, b, b, b};
    }
#pragma unroll
    for (int k = 0; k < kIn; k += 4) {
        const float a = X[row0 + lc][k + lr];
#pragma unroll
        for (int c = 0; c < 4; ++c) h1[c] = mfma4(a, W1[k + lr][16 * c + lc], h1[c]);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            h1[c][r] = in[r] ? tanhf(h1[c][r]) : 0.0f;
            A[row0 + 4 * lr + r][16 * c + lc] = h1[c][r];
        }
    __syncthreads();
    // layer 2: h2 = tanh(b2 + h1 W2)
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const float b = b2[16 * c + lc];
        h2[c] = f32x4{b, b, b, b};
    }
#pragma unroll 4
    for (int k = 0; k < kH; k += 4) {
        const float a = A[row0 + lc][k + lr];
#pragma unroll
        for (int c = 0; c < 4; ++c) h2[c] = mfma4(a, W2[k + lr][16 * c + lc], h2[c]);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            h2[c][r] = in[r] ? tanhf(h2[c][r]) : 0.0f;
            H[row0 + 4 * lr + r][16 * c + lc] = h2[c][r];
        }
    __syncthreads();
    // y = b3 + h2 w3, in every column; then d2 = dy w3 (1 - h2^2)
    f32x4 y = {b3, b3, b3, b3};
#pragma unroll 4
    for (int k = 0; k < kH; k += 4) y = mfma4(H[row0 + lc][k + lr], w3[k + lr], y);
    float dy[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int row = row0 + 4 * lr + r;
        const float e = y[r] - st[row];
        float l;
        if (nm.quantile > 0.0f) {
            const float q = e > 0.0f ? 1.0f - nm.quantile : -nm.quantile;
            dy[r] = q * scale;
            l = q * e * scale;
        } else {
            dy[r] = e * scale;
            l = 0.5f * e * e * scale;
        }
        if (!in[r]) dy[r] = l = 0.0f;
        if (lc == 0) {
            sdy[row] = dy[r];
            sloss[row] = l;
        }
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const float wc = w3[16 * c + lc];
#pragma unroll
        for (int r = 0; r < 4; ++r)
            B[row0 + 4 * lr + r][16 * c + lc] = dy[r] * wc * (1.0f - h2[c][r] * h2[c][r]);
    }
    __syncthreads();
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    float* out = part + (size_t)blockIdx.x * (kNParam + 1);
    // sums over the samples: W2's rows 16 w .. (h1_i d2_j), b2's and w3's columns
    // 16 w .. (d2_j, dy h2_j); wave 0 also dy and the loss
    {
        f32x4 g[4] = {zero, zero, zero, zero}, gb = zero, gw = zero, gs = zero;
#pragma unroll 4
        for (int k = 0; k < kGradRows; k += 4) {
            const float a = A[k + lr][row0 + lc];
#pragma unroll
            for (int c = 0; c < 4; ++c) g[c] = mfma4(a, B[k + lr][16 * c + lc], g[c]);
            gb = mfma4(1.0f, B[k + lr][row0 + lc], gb);
            gw = mfma4(sdy[k + lr], H[k + lr][row0 + lc], gw);
            if (w == 0) gs = mfma4(1.0f, lc == 0 ? sdy[k + lr] : (lc == 1 ? sloss[k + lr] : 0.0f), gs);
        }
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int r = 0; r < 4; ++r) out[kOffW2 + (row0 + 4 * lr + r) * kH + 16 * c + lc] = g[c][r];
        if (lr == 0) {
            out[kOffB2 + row0 + lc] = gb[0];
            out[kOffW3 + row0 + lc] = gw[0];
            if (w == 0 && lc < 2) out[lc == 0 ? kOffB3 : kNParam] = gs[0];
        }
    }
    // d1 = (W2 d2) (1 - h1^2), rows of this wave
    f32x4 d1[4] = {zero, zero, zero, zero};
#pragma unroll 4
    for (int k = 0; k < kH; k += 4) {
        const float a = B[row0 + lc][k + lr];
#pragma unroll
        for (int c = 0; c < 4; ++c) d1[c] = mfma4(a, W2[16 * c + lc][k + lr], d1[c]);
    }
    __syncthreads();   // every wave is done with h1 in A
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int r = 0; r < 4; ++r) A[row0 + 4 * lr + r][16 * c + lc] = d1[c][r] * (1.0f - h1[c][r] * h1[c][r]);
    __syncthreads();
    // W1's and b1's columns 16 w ..: sums of x_i d1_j and d1_j
    f32x4 g1 = zero, gb1 = zero;
#pragma unroll 4
    for (int k = 0; k < kGradRows; k += 4) {
        const float b = A[k + lr][row0 + lc];
        g1 = mfma4(X[k + lr][lc], b, g1);
        gb1 = mfma4(1.0f, b, gb1);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
        if (4 * lr + r < kIn) out[kOffW1 + (4 * lr + r) * kH + row0 + lc] = g1[r];
    if (lr == 0) out[kOffB1 + row0 + lc] = gb1[0];
}

// Sums per-block partials in block order: out[k] = sum_b part[b][k].  A block
// takes 64 parameters; its four waves fetch kReduceRows partials at a time into
// registers and then LDS, a round ahead of wave 0, which adds them in order.
// (One thread per parameter, loading and adding one after the other, took 72 us
// for 313 partials, this 4.9.)
constexpr uint32_t kReduceRows = 64;
__global__ __launch_bounds__(256) void k_mlp_reduce(const float* __restrict__ part, uint32_t nblk,
                                                    float* __restrict__ out)
{
    __shared__ float rows[2][kReduceRows][64];
    constexpr uint32_t kOwn = kReduceRows / 4;   // rows of a round per wave
    const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
    const uint32_t k = blockIdx.x * 64u + lane;
    const uint32_t kc = min(k, (uint32_t)kNParam);
    float v[kOwn];
    auto load = [&](uint32_t b0) {
#pragma unroll
        for (uint32_t u = 0; u < kOwn; ++u)
            v[u] = part[(size_t)min(b0 + w * kOwn + u, nblk - 1) * (kNParam + 1) + kc];
    };
    load(0);
    float a = 0.0f;
    for (uint32_t b0 = 0, h = 0; b0 < nblk; b0 += kReduceRows, h ^= 1u) {
#pragma unroll
        for (uint32_t u = 0; u < kOwn; ++u) rows[h][w * kOwn + u][lane] = v[u];
        load(b0 + kReduceRows);
        __syncthreads();
        if (w == 0) {
            const uint32_t cnt = min(kReduceRows, nblk - b0);
#pragma unroll 16
            for (uint32_t u = 0; u < cnt; ++u) a += rows[h][u][lane];
        }
    }
    if (w == 0 && k <= (uint32_t)kNParam) out[k] = a;
}

// Adam on the FP32 master weights, then the BF16 working copy.
__global__ void k_mlp_adam(float* __restrict__ w, float* __restrict__ m, float* __restrict__ v,
                           const float* __restrict__ g, uint16_t* __restrict__ wb, float lr, float b1, float b2,
                           float c1, float c2)
{
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= (uint32_t)kNParam) return;
    const float gk = g[k];
    const float mk = b1 * m[k] + (1.0f - b1) * gk;
    const float vk = b2 * v[k] + (1.0f - b2) * gk * gk;
    m[k] = mk;
    v[k] = vk;
    const float wk = w[k] - lr * (mk / c1) / (sqrtf(vk / c2) + 1e-8f);
    w[k] = wk;
    wb[k] = f32_to_bf16(wk);
}

__global__ void k_to_bf16(const float* __restrict__ w, uint16_t* __restrict__ wb, uint32_t n)
{
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) wb[k] = f32_to_bf16(w[k]);
}

}  // namespace rdamd

using namespace rdamd;

struct rd_mlp {
    int device = 0;
    hipStream_t stream = nullptr;
    float *w = nullptr, *m = nullptr, *v = nullptr, *g = nullptr, *part = nullptr;
    uint16_t* wb = nullptr;
    size_t part_blocks = 0;
    float *dx = nullptr, *dt = nullptr, *dy = nullptr;
    uint32_t* didx = nullptr;
    size_t cap = 0;
    Norm nm{};
    uint64_t adam_t = 0;
    std::mt19937 rng;
};

namespace {
thread_local std::string g_mlp_err;
int mfail(int code, const std::string& s)
{
    g_mlp_err = s;
    rdamd::set_last_error(s);
    return code;
}
#define MLP_TRY(expr)                                                                                   \
    do {                                                                                                \
        hipError_t e_ = (expr);                                                                         \
        if (e_ != hipSuccess) return mfail(RD_EDEVICE, std::string(#expr) + ": " + hipGetErrorString(e_)); \
    } while (0)

int ensure_cap(rd_mlp* p, size_t n)
{
    if (n <= p->cap) return RD_OK;
    if (p->dx) (void)hipFree(p->dx);
    if (p->dt) (void)hipFree(p->dt);
    if (p->dy) (void)hipFree(p->dy);
    if (p->didx) (void)hipFree(p->didx);
    MLP_TRY(hipMalloc((void**)&p->dx, n * kIn * sizeof(float)));
    MLP_TRY(hipMalloc((void**)&p->dt, n * sizeof(float)));
    MLP_TRY(hipMalloc((void**)&p->dy, n * sizeof(float)));
    MLP_TRY(hipMalloc((void**)&p->didx, n * sizeof(uint32_t)));
    p->cap = n;
    return RD_OK;
}
int ensure_part(rd_mlp* p, size_t nblk)
{
    if (nblk <= p->part_blocks) return RD_OK;
    if (p->part) (void)hipFree(p->part);
    MLP_TRY(hipMalloc((void**)&p->part, nblk * (kNParam + 1) * sizeof(float)));
    p->part_blocks = nblk;
    return RD_OK;
}
}  // namespace

namespace rdamd {
const uint16_t* mlp_weights(const rd_mlp* p) { return p->wb; }
int mlp_device(const rd_mlp* p) { return p->device; }
int mlp_forward_dev(const rd_mlp* p, hipStream_t st, const float* x, uint32_t n, float* y)
{
    if (n == 0) return RD_OK;
    hipLaunchKernelGGL(k_mlp_forward, dim3(n), dim3(kH), 0, st, p->wb, p->nm, x, n, y);
    return hipGetLastError() == hipSuccess ? RD_OK : RD_EDEVICE;
}
}  // namespace rdamd

extern "C" {

int rd_mlp_create(int device, uint32_t seed, rd_mlp** out)
{
    DeviceScope dev_scope(device);
    if (!out) return mfail(RD_EINVAL, "NULL argument");
    rd_mlp* p = new rd_mlp();
    p->device = device;
    p->rng.seed(seed);
    hipError_t e = hipSetDevice(device);
    if (e == hipSuccess) e = hipStreamCreateWithFlags(&p->stream, hipStreamNonBlocking);
    if (e != hipSuccess) {
        delete p;
        return mfail(RD_EDEVICE, std::string("rd_mlp_create: ") + hipGetErrorString(e));
    }
    e = hipMalloc((void**)&p->w, kNParam * sizeof(float));
    if (e == hipSuccess) e = hipMalloc((void**)&p->m, kNParam * sizeof(float));
    if (e == hipSuccess) e = hipMalloc((void**)&p->v, kNParam * sizeof(float));
    if (e == hipSuccess) e = hipMalloc((void**)&p->g, (kNParam + 1) * sizeof(float));
    if (e == hipSuccess) e = hipMalloc((void**)&p->wb, kNParam * sizeof(uint16_t));
    if (e != hipSuccess) {
        rd_mlp_destroy(p);
        return mfail(RD_ENOMEM, std::string("rd_mlp_create: hipMalloc: ") + hipGetErrorString(e));
    }
    // Glorot-uniform weights, zero biases
    std::vector<float> w(kNParam, 0.0f);
    auto fill = [&](int off, int fan_in, int fan_out, int count) {
        const float lim = std::sqrt(6.0f / (fan_in + fan_out));
        std::uniform_real_distribution<float> u(-lim, lim);
        for (int k = 0; k < count; ++k) w[off + k] = u(p->rng);
    };
    fill(kOffW1, kIn, kH, kIn * kH);
    fill(kOffW2, kH, kH, kH * kH);
    fill(kOffW3, kH, 1, kH);
    for (int i = 0; i < kIn; ++i) { p->nm.mean[i] = 0.0f; p->nm.inv_std[i] = 1.0f; }
    p->nm.t_mean = 0.0f;
    p->nm.t_std = 1.0f;
    p->nm.base = -1;
    p->nm.quantile = 0.0f;
    if (int rc = rd_mlp_set_params(p, w.data())) {
        rd_mlp_destroy(p);
        return rc;
    }
    *out = p;
    return RD_OK;
}

int rd_mlp_destroy(rd_mlp* p)
{
    DeviceScope dev_scope(p ? p->device : -1);
    if (!p) return RD_OK;
    (void)hipStreamSynchronize(p->stream);
    for (void* q : {(void*)p->w, (void*)p->m, (void*)p->v, (void*)p->g, (void*)p->wb, (void*)p->part, (void*)p->dx,
                    (void*)p->dt, (void*)p->dy, (void*)p->didx})
        if (q) (void)hipFree(q);
    (void)hipStreamDestroy(p->stream);
    delete p;
    return RD_OK;
}

int rd_mlp_set_norm(rd_mlp* p, const float mean[RD_MLP_IN], const float stdev[RD_MLP_IN], float t_mean, float t_std)
{
    DeviceScope dev_scope(p ? p->device : -1);
    if (!p || !mean || !stdev || !(t_std > 0.0f)) return mfail(RD_EINVAL, "bad argument");
    for (int i = 0; i < kIn; ++i) {
        if (!(stdev[i] > 0.0f)) return mfail(RD_EINVAL, "feature std must be > 0");
        p->nm.mean[i] = mean[i];
        p->nm.inv_std[i] = 1.0f / stdev[i];
    }
    p->nm.t_mean = t_mean;
    p->nm.t_std = t_std;
    return RD_OK;
}

int rd_mlp_set_target(rd_mlp* p, int base_feature, float quantile)
{
    if (!p) return mfail(RD_EINVAL, "NULL model");
    if (base_feature < -1 || base_feature >= kIn) return mfail(RD_EINVAL, "base feature must be -1 or 0..11");
    if (!(quantile == 0.0f || (quantile > 0.0f && quantile < 1.0f)))
        return mfail(RD_EINVAL, "quantile must be 0 (mean) or in (0, 1)");
    p->nm.base = base_feature;
    p->nm.quantile = quantile;
    return RD_OK;
}

int rd_mlp_set_params(rd_mlp* p, const float* params)
{
    DeviceScope dev_scope(p ? p->device : -1);
    if (!p || !params) return mfail(RD_EINVAL, "bad argument");
    MLP_TRY(hipMemcpyAsync(p->w, params, kNParam * sizeof(float), hipMemcpyHostToDevice, p->stream));
    MLP_TRY(hipMemsetAsync(p->m, 0, kNParam * sizeof(float), p->stream));
    MLP_TRY(hipMemsetAsync(p->v, 0, kNParam * sizeof(float), p->stream));
    hipLaunchKernelGGL(k_to_bf16, dim3((kNParam + 255) / 256), dim3(256), 0, p->stream, p->w, p->wb,
                       (uint32_t)kNParam);
    MLP_TRY(hipGetLastError());
    MLP_TRY(hipStreamSynchronize(p->stream));
    p->adam_t = 0;
    return RD_OK;
}

int rd_mlp_get_params(rd_mlp* p, float* params, uint16_t* params_bf16)
{
    DeviceScope dev_scope(p ? p->device : -1);
    if (!p) return mfail(RD_EINVAL, "bad argument");
    if (params) MLP_TRY(hipMemcpyAsync(params, p->w, kNParam * sizeof(float), hipMemcpyDeviceToHost, p->stream));
    if (params_bf16)
        MLP_TRY(hipMemcpyAsync(params_bf16, p->wb, kNParam * sizeof(uint16_t), hipMemcpyDeviceToHost, p->stream));
    MLP_TRY(hipStreamSynchronize(p->stream));
    return RD_OK;
}

int rd_mlp_forward(rd_mlp* p, const float* x, uint32_t n, float* y)
{
    DeviceScope dev_scope(p ? p->device : -1);
    if (!p || (!x && n) || (!y && n)) return mfail(RD_EINVAL, "bad argument");
    if (n == 0) return RD_OK;
    if (int rc = ensure_cap(p, n)) return rc;
    MLP_TRY(hipMemcpyAsync(p->dx, x, (size_t)n * kIn * sizeof(float), hipMemcpyHostToDevice, p->stream));
    if (int rc = mlp_forward_dev(p, p->stream, p->dx, n, p->dy)) return mfail(rc, "k_mlp_forward launch");
    MLP_TRY(hipMemcpyAsync(y, p->dy, n * sizeof(float), hipMemcpyDeviceToHost, p->stream));
    MLP_TRY(hipStreamSynchronize(p->stream));
    return RD_OK;
}

static int grad_dev(rd_mlp* p, const uint32_t* idx, uint32_t n, float scale)
{
    const uint32_t nblk = (n + kGradRows - 1) / kGradRows;
    if (int rc = ensure_part(p, nblk)) return rc;
    hipLaunchKernelGGL(k_mlp_grad, dim3(nblk), dim3(kGradBlock), 0, p->stream, p->wb, p->nm, p->dx, p->dt, idx, n,
                       scale, p->part);
    MLP_TRY(hipGetLastError());
    hipLaunchKernelGGL(k_mlp_reduce, dim3((kNParam + 1 + 63) / 64), dim3(256), 0, p->stream, p->part, nblk, p->g);
    MLP_TRY(hipGetLastError());
    return RD_OK;
}

int rd_mlp_loss_grad(rd_mlp* p, const float* x, const float* t, uint32_t n, float* loss, float* grad)
{
    DeviceScope dev_scope(p ? p->device : -1);
    if (!p || !x || !t || n == 0) return mfail(RD_EINVAL, "bad argument");
    if (int rc = ensure_cap(p, n)) return rc;
    MLP_TRY(hipMemcpyAsync(p->dx, x, (size_t)n * kIn * sizeof(float), hipMemcpyHostToDevice, p->stream));
    MLP_TRY(hipMemcpyAsync(p->dt, t, n * sizeof(float), hipMemcpyHostToDevice, p->stream));
    if (int rc = grad_dev(p, nullptr, n, 1.0f / n)) return rc;
    std::vector<float> g(kNParam + 1);
    MLP_TRY(hipMemcpyAsync(g.data(), p->g, (kNParam + 1) * sizeof(float), hipMemcpyDeviceToHost, p->stream));
    MLP_TRY(hipStreamSynchronize(p->stream));
    if (grad) std::memcpy(grad, g.data(), kNParam * sizeof(float));
    if (loss) *loss = g[kNParam];
    return RD_OK;
}

int rd_mlp_train(rd_mlp* p, const float* x, const float* t, uint32_t n, uint32_t epochs, uint32_t batch, float lr,
                 float* final_loss)
{
    DeviceScope dev_scope(p ? p->device : -1);
    if (!p || !x || !t || n == 0 || batch == 0) return mfail(RD_EINVAL, "bad argument");
    if (int rc = ensure_cap(p, n)) return rc;
    MLP_TRY(hipMemcpyAsync(p->dx, x, (size_t)n * kIn * sizeof(float), hipMemcpyHostToDevice, p->stream));
    MLP_TRY(hipMemcpyAsync(p->dt, t, n * sizeof(float), hipMemcpyHostToDevice, p->stream));
    std::vector<uint32_t> perm(n);
    for (uint32_t i = 0; i < n; ++i) perm[i] = i;
    const float b1 = 0.9f, b2 = 0.999f;
    double last = 0.0;
    for (uint32_t ep = 0; ep < epochs; ++ep) {
        std::shuffle(perm.begin(), perm.end(), p->rng);
        MLP_TRY(hipMemcpyAsync(p->didx, perm.data(), n * sizeof(uint32_t), hipMemcpyHostToDevice, p->stream));
        double ep_loss = 0.0;
        std::vector<float> lbuf;
        for (uint32_t s = 0; s < n; s += batch) {
            const uint32_t nb = std::min(batch, n - s);
            if (int rc = grad_dev(p, p->didx + s, nb, 1.0f / nb)) return rc;
            p->adam_t++;
            const float c1 = 1.0f - std::pow(b1, (float)p->adam_t), c2 = 1.0f - std::pow(b2, (float)p->adam_t);
            hipLaunchKernelGGL(k_mlp_adam, dim3((kNParam + 255) / 256), dim3(256), 0, p->stream, p->w, p->m, p->v,
                               p->g, p->wb, lr, b1, b2, c1, c2);
            MLP_TRY(hipGetLastError());
            if (ep + 1 == epochs) {
                float l;
                MLP_TRY(hipMemcpyAsync(&l, p->g + kNParam, sizeof(float), hipMemcpyDeviceToHost, p->stream));
                MLP_TRY(hipStreamSynchronize(p->stream));
                ep_loss += (double)l * nb;
            }
        }
        MLP_TRY(hipStreamSynchronize(p->stream));
        last = ep_loss / n;
    }
    if (final_loss) *final_loss = (float)last;
    return RD_OK;
}

}  // extern "C"
