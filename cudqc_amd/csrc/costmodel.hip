// HIP kernels of the subtree-cost model (forward, full-data gradient, Adam training)
// and their C-ABI (include/dqc.h). The model orders and splits the task batches of the
// learned schedule; it changes only the order in which tasks run, never the output.
//
// Training is deterministic: each workgroup takes chunks of 64 samples through the network
// on matrix cores, accumulates its weight gradients in registers, and the partial gradients
// are summed in a fixed order by the kernel that applies the Adam step.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <random>
#include <vector>

#include "../../include/dqc.h"
#include "costmodel.hpp"
#include "devpool.hpp"

namespace {

using namespace dqc_cost;

constexpr int GT = 256;                              // threads per training workgroup
constexpr int CH = 64;                               // samples per chunk
constexpr int MAX_BLOCKS = 512;

static_assert(NPARAM == DQC_MLP_PARAMS, "parameter count");
static_assert(IN == DQC_MLP_IN && H == DQC_MLP_HIDDEN, "model shape");

// The network on matrix cores in fp32 (v_mfma_f32_16x16x4: operand and result layout of the
// CDNA ISA). A wavefront takes 16 samples: units are rows and samples columns, so lane l
// holds sample l % 16 and, in register 4 t + r, unit 16 t + 4 (l / 16) + r. A layer's result has
// the layout in which the next product takes it as its right operand, with the units summed
// in the order (t, r), so activations never leave the registers between layers.
typedef float f4 __attribute__((ext_vector_type(4)));
constexpr int LDW = H + 1;  // row stride of a 64-wide LDS matrix (banks)
struct Act { f4 v[4]; };     // 64 units x 16 samples
__device__ __forceinline__ float relu(float z) { return z > 0.f ? z : 0.f; }
__device__ __forceinline__ int unit_of(int t, int r, int lane) { return 16 * t + 4 * (lane >> 4) + r; }
__device__ __forceinline__ Act unit_values(const float* p, int lane) {  // p[unit], for each of the lane's units
    Act a;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) a.v[t][r] = p[unit_of(t, r, lane)];
    return a;
}
// acc[u] (rows 16 u ..) += A (64 x 64) * B, A's operand given by a(u, k) with k = 4 t + r standing
// for column unit_of(t, r, lane) of row 16 u + lane % 16
template <class F>
__device__ __forceinline__ void mul64(Act& acc, const Act& B, F&& a) {
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int u = 0; u < 4; ++u)
                acc.v[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(a(u, 4 * t + r), B.v[t][r], acc.v[u], 0, 0, 0);
}
// First layer before its ReLU: z = b1 + W1 x, the 7 features padded to 8. x0 / x1: features
// lane / 16 and 4 + lane / 16 of the lane's sample.
__device__ __forceinline__ Act layer1(const float* p, const Act& b1, float x0, float x1, int lane) {
    Act z = b1;
    const int k = lane >> 4;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const float* w = p + OFF_W1 + (16 * u + (lane & 15)) * IN;
        z.v[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[k], x0, z.v[u], 0, 0, 0);
        z.v[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(k < 3 ? w[4 + k] : 0.f, x1, z.v[u], 0, 0, 0);
    }
    return z;
}
__device__ __forceinline__ Act relu(Act a) {
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) a.v[t][r] = relu(a.v[t][r]);
    return a;
}
// sum over the lane's units of w * b, then over the four lanes of its sample
__device__ __forceinline__ float head(const Act& w, const Act& b, float b3) {
    float y = 0.f;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) y += w.v[t][r] * b.v[t][r];
    y += __shfl_xor(y, 16, 64);
    y += __shfl_xor(y, 32, 64);
    return y + b3;
}

// y = the network's prediction for n samples. Bound by the fp32 matrix rate: 72 products of
// 16x16x4 a wavefront per 16 samples; the second layer's weights stay in registers.
// 262,144 samples: 37 us (one sample per thread, weights in LDS: 195 us).
__global__ __launch_bounds__(256) void forward_kernel(const float* __restrict__ params, const float* __restrict__ x,
                                                      long long n, float* __restrict__ y) {
    __shared__ float p[NPARAM];
    for (int i = threadIdx.x; i < NPARAM; i += blockDim.x) p[i] = params[i];
    __syncthreads();
    const int lane = threadIdx.x & 63;
    const Act b1 = unit_values(p + OFF_B1, lane), b2 = unit_values(p + OFF_B2, lane), w3 = unit_values(p + OFF_W3, lane);
    float w2[4][16];
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int k = 0; k < 16; ++k)
            w2[u][k] = p[OFF_W2 + (16 * u + (lane & 15)) * H + unit_of(k >> 2, k & 3, lane)];
    const float b3 = p[OFF_B3];
    const long long waves = (long long)gridDim.x * (blockDim.x >> 6);
    for (long long s0 = ((long long)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) * 16; s0 < n; s0 += 16 * waves) {
        const long long s = s0 + (lane & 15);
        const int k = lane >> 4;
        const float x0 = s < n ? x[IN * s + k] : 0.f, x1 = s < n && k < 3 ? x[IN * s + 4 + k] : 0.f;
        const Act a = relu(layer1(p, b1, x0, x1, lane));
        Act z = b2;
        mul64(z, a, [&](int u, int k2) { return w2[u][k2]; });
        const float v = head(w3, relu(z), b3);
        if (lane < 16 && s < n) y[s] = v;
    }
}

// Gradient of sum_s scale * (y_s - t_s)^2 over samples idx[0..m) (idx null: 0..m-1).
// partial[block][p] gets the block's share, lpart[block] its sum of squared errors (GRAD
// false: only that). Each of the four wavefronts takes 16 samples of a chunk through both
// passes in registers; the weight gradients are products over the chunk's 64 samples, whose
// activations and pre-activation gradients meet in LDS, and stay in accumulators over the
// block's chunks. Bound by latency at a training batch (1,024 samples are 16 workgroups of one
// chunk): 17 us a call there, 58 us with vector instructions.
template <bool GRAD>
__global__ __launch_bounds__(GT, 1) void grad_kernel(const float* __restrict__ params, const float* __restrict__ x,
                                                     const float* __restrict__ t, const int32_t* __restrict__ idx,
                                                     long long m, float scale, float* __restrict__ partial,
                                                     double* __restrict__ lpart) {
    __shared__ float p[NPARAM];
    __shared__ float A[H * LDW];  // [unit][sample]: first hidden layer
    __shared__ float B[H * LDW];  // pre-activation gradient of the second hidden layer
    __shared__ float C[H * LDW];  // and of the first
    __shared__ float X[8 * LDW];  // [feature][sample], feature 7 = 1 (the bias)
    __shared__ double lred[GT];
    __shared__ float red[2][4][H];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, col = lane & 15, k = lane >> 4;
    for (int i = tid; i < NPARAM; i += GT) p[i] = params[i];
    __syncthreads();
    const Act b1 = unit_values(p + OFF_B1, lane), b2 = unit_values(p + OFF_B2, lane), w3 = unit_values(p + OFF_W3, lane);
    const float b3 = p[OFF_B3];
    f4 g2[4] = {}, g1 = {};   // this wavefront's rows 16 wave .. of dW2 (4 column tiles) and of dW1 | db1
    Act gw3 = {}, gb2 = {};
    float gb3 = 0.f;
    double loss = 0.0;
    const long long nchunk = (m + CH - 1) / CH;
    for (long long c = blockIdx.x; c < nchunk; c += gridDim.x) {
        const long long s = c * CH + 16 * wave + col;
        const bool live = s < m;
        const long long at = live ? (idx ? (long long)idx[s] : s) : 0;
        const float x0 = live ? x[at * IN + k] : 0.f, x1 = live && k < 3 ? x[at * IN + 4 + k] : 0.f;
        const Act a = relu(layer1(p, b1, x0, x1, lane));
        Act z = b2;
        mul64(z, a, [&](int u, int kk) { return p[OFF_W2 + (16 * u + col) * H + unit_of(kk >> 2, kk & 3, lane)]; });
        const Act b = relu(z);
        const float r = live ? head(w3, b, b3) - t[at] : 0.f;
        if (lane < 16) loss += (double)r * (double)r;
        if (!GRAD) continue;
        const float dy = 2.f * scale * r;
        if (lane < 16) gb3 += dy;
        Act db;
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                gw3.v[q][e] += dy * b.v[q][e];
                db.v[q][e] = b.v[q][e] > 0.f ? dy * w3.v[q][e] : 0.f;
                gb2.v[q][e] += db.v[q][e];
            }
        Act da = {};
        mul64(da, db, [&](int u, int kk) { return p[OFF_W2 + unit_of(kk >> 2, kk & 3, lane) * H + 16 * u + col]; });
        __syncthreads();  // (the previous chunk's products are done with the LDS matrices)
        const int sc = 16 * wave + col;
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int u = unit_of(q, e, lane);
                A[u * LDW + sc] = a.v[q][e];
                B[u * LDW + sc] = db.v[q][e];
                C[u * LDW + sc] = a.v[q][e] > 0.f ? da.v[q][e] : 0.f;
            }
        X[k * LDW + sc] = x0;
        X[(4 + k) * LDW + sc] = k < 3 ? x1 : live ? 1.f : 0.f;
        __syncthreads();
        const int row = 16 * wave + col;
#pragma unroll 4
        for (int kb = 0; kb < CH / 4; ++kb) {
            const int ss = 4 * kb + k;
            const float fb = B[row * LDW + ss], fc = C[row * LDW + ss];
#pragma unroll
            for (int u = 0; u < 4; ++u)
                g2[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(fb, A[(16 * u + col) * LDW + ss], g2[u], 0, 0, 0);
            g1 = __builtin_amdgcn_mfma_f32_16x16x4f32(fc, col < 8 ? X[col * LDW + ss] : 0.f, g1, 0, 0, 0);
        }
    }
    if (GRAD) {
        float* out = partial + (long long)blockIdx.x * NPARAM;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int j = 16 * wave + 4 * k + e;
#pragma unroll
            for (int u = 0; u < 4; ++u) out[OFF_W2 + j * H + 16 * u + col] = g2[u][e];
            if (col < IN) out[OFF_W1 + j * IN + col] = g1[e];
            else if (col == IN) out[OFF_B1 + j] = g1[e];
        }
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float w = gw3.v[q][e], v = gb2.v[q][e];
                for (int off = 8; off > 0; off >>= 1) {  // over the wavefront's 16 samples
                    w += __shfl_xor(w, off, 64);
                    v += __shfl_xor(v, off, 64);
                }
                if (col == 0) {
                    red[0][wave][unit_of(q, e, lane)] = w;
                    red[1][wave][unit_of(q, e, lane)] = v;
                }
            }
        for (int off = 8; off > 0; off >>= 1) gb3 += __shfl_xor(gb3, off, 64);
    }
    lred[tid] = loss;
    __syncthreads();
    if (GRAD) {
        float* out = partial + (long long)blockIdx.x * NPARAM;
        if (tid < 2 * H) {
            const int q = tid / H, j = tid % H;
            out[(q ? OFF_B2 : OFF_W3) + j] = red[q][0][j] + red[q][1][j] + red[q][2][j] + red[q][3][j];
        }
        __syncthreads();
        if (lane == 0) red[0][wave][0] = gb3;
        __syncthreads();
        if (tid == 0) out[OFF_B3] = red[0][0][0] + red[0][1][0] + red[0][2][0] + red[0][3][0];
    }
    if (tid == 0) {
        double sum = 0.0;
        for (int w = 0; w < 4; ++w)
            for (int i = 0; i < 16; ++i) sum += lred[64 * w + i];  // (a sample's error is in its first lane)
        lpart[blockIdx.x] = sum;
    }
}

// grad[q] = sum over blocks of partial[b][q], in block order.
__global__ void reduce_kernel(const float* __restrict__ partial, int nblocks, float* __restrict__ grad) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= NPARAM) return;
    float g = 0.f;
    for (int b = 0; b < nblocks; ++b) g += partial[(long long)b * NPARAM + q];
    grad[q] = g;
}

// One Adam step on the blocks' partial gradients (summed in block order, as reduce_kernel
// does): one launch instead of two, bound by its latency.
__global__ void adam_kernel(float* __restrict__ p, const float* __restrict__ partial, int nblocks, float* __restrict__ mo,
                            float* __restrict__ ve, float lr, float c1, float c2) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= NPARAM) return;
    float g = 0.f;
#pragma unroll 8
    for (int b = 0; b < nblocks; ++b) g += partial[(long long)b * NPARAM + q];
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    const float m = b1 * mo[q] + (1.f - b1) * g;
    const float v = b2 * ve[q] + (1.f - b2) * g * g;
    mo[q] = m;
    ve[q] = v;
    p[q] -= lr * (m / c1) / (sqrtf(v / c2) + eps);
}

// Device buffers of one call; given back on scope exit, when nothing queued uses them.
struct Buf {
    std::vector<std::pair<void*, size_t>> ptrs;
    ~Buf() {
        if (!ptrs.empty()) hipStreamSynchronize(nullptr);
        for (auto& q : ptrs) dqc::DevicePool::get().give(q.first, q.second);
    }
    template <class T>
    T* alloc(size_t count) {
        void* q = nullptr;
        const size_t bytes = std::max<size_t>(count, 1) * sizeof(T);
        if (dqc::DevicePool::get().take(&q, bytes) != hipSuccess) return nullptr;
        ptrs.push_back({q, bytes});
        return (T*)q;
    }
};

int grad_blocks(long long m) {
    return (int)std::max<long long>(1, std::min<long long>(MAX_BLOCKS, (m + CH - 1) / CH));
}

// Full-data gradient (dgrad null: only the error) on device buffers; gives the sum of squared
// errors.
bool device_gradient(const float* dp, const float* dx, const float* dt, long long n, float* dgrad, float* dpart,
                     double* dl, double* sse) {
    const int nb = grad_blocks(n);
    if (dgrad) {
        grad_kernel<true><<<nb, GT>>>(dp, dx, dt, nullptr, n, 1.f / (float)n, dpart, dl);
        reduce_kernel<<<(NPARAM + 255) / 256, 256>>>(dpart, nb, dgrad);
    } else {
        grad_kernel<false><<<nb, GT>>>(dp, dx, dt, nullptr, n, 1.f / (float)n, dpart, dl);
    }
    std::vector<double> l(nb);
    if (hipMemcpy(l.data(), dl, sizeof(double) * nb, hipMemcpyDeviceToHost) != hipSuccess) return false;
    double s = 0.0;
    for (double v : l) s += v;
    *sse = s;
    return hipGetLastError() == hipSuccess;
}

}  // namespace

extern "C" {

dqc_status dqc_task_features(const dqc_task_log* r, int64_t n, float* x) {
    if (n < 0 || (n > 0 && (!r || !x))) return DQC_E_ARG;
    for (int64_t i = 0; i < n; ++i)
        features(r[i].nm, r[i].tot, r[i].depth, r[i].dmin_out, r[i].dmax_out, r[i].dmin_in, r[i].dmax_in, x + IN * i);
    return DQC_OK;
}

dqc_status dqc_mlp_forward(const float* params, const float* x, int64_t n, float* y) {
    if (!params || n < 0 || (n > 0 && (!x || !y))) return DQC_E_ARG;
    if (n == 0) return DQC_OK;
    Buf b;
    float *dp = b.alloc<float>(NPARAM), *dx = b.alloc<float>((size_t)n * IN), *dy = b.alloc<float>((size_t)n);
    if (!dp || !dx || !dy) return DQC_E_HIP;
    if (hipMemcpy(dp, params, sizeof(float) * NPARAM, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(dx, x, sizeof(float) * IN * (size_t)n, hipMemcpyHostToDevice) != hipSuccess)
        return DQC_E_HIP;
    const int blocks = (int)std::min<long long>(768, (n + 63) / 64);  // three workgroups a CU, 16 samples a wavefront
    forward_kernel<<<blocks, 256>>>(dp, dx, n, dy);
    if (hipGetLastError() != hipSuccess ||
        hipMemcpy(y, dy, sizeof(float) * (size_t)n, hipMemcpyDeviceToHost) != hipSuccess)
        return DQC_E_HIP;
    return DQC_OK;
}

dqc_status dqc_mlp_gradient(const float* params, const float* x, const float* t, int64_t n, float* grad,
                            double* loss) {
    if (!params || !grad || n <= 0 || !x || !t) return DQC_E_ARG;
    Buf b;
    const int nb = grad_blocks(n);
    float *dp = b.alloc<float>(NPARAM), *dx = b.alloc<float>((size_t)n * IN), *dt = b.alloc<float>((size_t)n);
    float *dg = b.alloc<float>(NPARAM), *dpart = b.alloc<float>((size_t)nb * NPARAM);
    double* dl = b.alloc<double>(nb);
    if (!dp || !dx || !dt || !dg || !dpart || !dl) return DQC_E_HIP;
    if (hipMemcpy(dp, params, sizeof(float) * NPARAM, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(dx, x, sizeof(float) * IN * (size_t)n, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(dt, t, sizeof(float) * (size_t)n, hipMemcpyHostToDevice) != hipSuccess)
        return DQC_E_HIP;
    double sse = 0.0;
    if (!device_gradient(dp, dx, dt, n, dg, dpart, dl, &sse)) return DQC_E_HIP;
    if (hipMemcpy(grad, dg, sizeof(float) * NPARAM, hipMemcpyDeviceToHost) != hipSuccess) return DQC_E_HIP;
    if (loss) *loss = sse / (double)n;
    return DQC_OK;
}

dqc_status dqc_mlp_train(float* params, const float* x, const float* t, int64_t n, int32_t epochs, int32_t batch,
                         float lr, uint64_t seed, double* loss) {
    if (!params || !x || !t || n <= 0 || epochs < 0 || batch < 1 || !(lr > 0.f) || n > INT32_MAX) return DQC_E_ARG;
    Buf b;
    const int nb = grad_blocks(std::min<long long>(n, batch));
    const int nbf = grad_blocks(n);
    float *dp = b.alloc<float>(NPARAM), *dx = b.alloc<float>((size_t)n * IN), *dt = b.alloc<float>((size_t)n);
    float *dm = b.alloc<float>(NPARAM), *dv = b.alloc<float>(NPARAM);
    float* dpart = b.alloc<float>((size_t)nb * NPARAM);
    double* dl = b.alloc<double>(std::max(nb, nbf));
    int32_t* didx = b.alloc<int32_t>((size_t)n);
    if (!dp || !dx || !dt || !dm || !dv || !dpart || !dl || !didx) return DQC_E_HIP;
    if (hipMemcpy(dp, params, sizeof(float) * NPARAM, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(dx, x, sizeof(float) * IN * (size_t)n, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(dt, t, sizeof(float) * (size_t)n, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemset(dm, 0, sizeof(float) * NPARAM) != hipSuccess || hipMemset(dv, 0, sizeof(float) * NPARAM) != hipSuccess)
        return DQC_E_HIP;
    std::vector<int32_t> order((size_t)n);
    for (int64_t i = 0; i < n; ++i) order[i] = (int32_t)i;
    std::mt19937_64 rng(seed);
    long long step = 0;
    for (int e = 0; e < epochs; ++e) {
        for (int64_t i = n - 1; i > 0; --i) {  // Fisher-Yates with a bounded draw
            const uint64_t r = rng() % (uint64_t)(i + 1);
            std::swap(order[i], order[r]);
        }
        if (hipMemcpy(didx, order.data(), sizeof(int32_t) * (size_t)n, hipMemcpyHostToDevice) != hipSuccess)
            return DQC_E_HIP;
        for (long long s0 = 0; s0 < n; s0 += batch) {
            const long long m = std::min<long long>(batch, n - s0);
            const int blocks = grad_blocks(m);
            grad_kernel<true><<<blocks, GT>>>(dp, dx, dt, didx + s0, m, 1.f / (float)m, dpart, dl);
            ++step;
            // (in double: 1 - 0.999^step cancels, and in float its error, 6e-5 at the first step, was
            // most of what training was off by)
            const float c1 = (float)(1.0 - std::pow((double)0.9f, (double)step));
            const float c2 = (float)(1.0 - std::pow((double)0.999f, (double)step));
            adam_kernel<<<(NPARAM + 63) / 64, 64>>>(dp, dpart, blocks, dm, dv, lr, c1, c2);
        }
        if (hipGetLastError() != hipSuccess) return DQC_E_HIP;
    }
    double sse = 0.0;
    if (!device_gradient(dp, dx, dt, n, nullptr, dpart, dl, &sse)) return DQC_E_HIP;
    if (hipMemcpy(params, dp, sizeof(float) * NPARAM, hipMemcpyDeviceToHost) != hipSuccess) return DQC_E_HIP;
    if (loss) *loss = sse / (double)n;
    return DQC_OK;
}

}  // extern "C"
