// Per-front update-precision classifier: a 16 -> 64 -> 64 -> 3 multilayer perceptron (ReLU
// hidden layers, softmax output over {BF16, FP32, FP64}), FP32, with its training on the GPU.
// The reference has no counterpart; the solver uses it to choose each front's Schur-update
// arithmetic from front features, with full FP64 as the fallback.
//
// Parameters, one FP32 array of RV_MLP_PARAMS entries: W1[16][64], b1[64], W2[64][64], b2[64],
// W3[64][3], b3[3] (row = input unit).  Training is full-batch Adam on the class-weighted mean
// cross-entropy L = sum_n w[y_n] (-log p[n][y_n]) / sum_n w[y_n].  Every reduction runs in a
// fixed order (samples within a workgroup's chunks, then the workgroups), so training is
// deterministic.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <map>
#include <mutex>
#include <stdexcept>
#include <string>
#include <vector>

#include "rv_mlp.h"

namespace rv {

namespace {

constexpr int NI = MLP_IN, NH = MLP_HID, NO = MLP_OUT;
constexpr int O_W1 = 0, O_B1 = O_W1 + NI * NH, O_W2 = O_B1 + NH, O_B2 = O_W2 + NH * NH, O_W3 = O_B2 + NH,
              O_B3 = O_W3 + NH * NO, NPAR = O_B3 + NO;
static_assert(NPAR == MLP_PARAMS, "parameter layout");

#define MLP_HIP(x)                                                                        \
    do {                                                                                  \
        hipError_t e_ = (x);                                                              \
        if (e_ != hipSuccess) throw std::runtime_error(std::string("HIP: ") + hipGetErrorString(e_)); \
    } while (0)

// Forward pass and gradient in one launch.  A workgroup takes 64 samples at a time through every
// layer with all activations in LDS: nothing but the features and labels is read and nothing but
// the probabilities or one partial gradient per workgroup written (one thread per sample for the
// passes and one per parameter, serial over the samples, for the gradient took 0.06 + 0.04 +
// 4.3 ms on 16738 samples; now 30 us and 5 for the reduction, 17 for the forward pass alone).
// The products run in register tiles of 4 x 4; the activations are stored with the samples
// consecutive (rows of SP = 64 + 4 floats: 16-byte reads, and rows of consecutive units start four
// banks apart).  Two workgroups per CU (80 KB of LDS); at most GRID workgroups, each summing its
// chunks' gradients in registers, so the partials stay within GRID rows for any sample count.
constexpr int SC = 64, SP = SC + 4, GRID = 512;
struct MlpLds {
    float W1[NI][NH], W2[NH][SP], W3[NH * NO], b1[NH], b2[NH], b3[4];
    float X[NI][SP], H1[NH][SP], H2[NH][SP], D1[NH][SP];  // H2 becomes the delta of layer 2
    float z[NO][SC], d3[NO][SC], loss[SC];
};

__device__ __forceinline__ void fma4(float (&acc)[4], float w, const float4 &v) {
    acc[0] = fmaf(w, v.x, acc[0]);
    acc[1] = fmaf(w, v.y, acc[1]);
    acc[2] = fmaf(w, v.z, acc[2]);
    acc[3] = fmaf(w, v.w, acc[3]);
}
__device__ __forceinline__ float dot4(float acc, const float4 &a, const float4 &b) {
    return fmaf(a.w, b.w, fmaf(a.z, b.z, fmaf(a.y, b.y, fmaf(a.x, b.x, acc))));
}
__device__ __forceinline__ float4 &row4(float *p) { return *reinterpret_cast<float4 *>(p); }

template <bool GRAD>
__global__ __launch_bounds__(256) void k_mlp(const float *__restrict__ par, int n, const float *__restrict__ x,
                                             const int *__restrict__ y, const float *__restrict__ cw, float inv_wsum,
                                             float *__restrict__ prob, float *__restrict__ part) {
    __shared__ __align__(16) MlpLds L;
    const int t = threadIdx.x;
    for (int i = t; i < NPAR; i += 256) {
        const float v = par[i];
        if (i < O_B1) L.W1[i / NH][i % NH] = v;
        else if (i < O_W2) L.b1[i - O_B1] = v;
        else if (i < O_B2) L.W2[(i - O_W2) / NH][(i - O_W2) % NH] = v;
        else if (i < O_W3) L.b2[i - O_B2] = v;
        else if (i < O_B3) L.W3[i - O_W3] = v;
        else L.b3[i - O_B3] = v;
    }
    const int tr = t >> 4, tc = t & 15;  // samples 4 tr .. 4 tr + 3, units tc + 16 b
    float g1[4] = {0, 0, 0, 0}, g2[4][4] = {}, g3 = 0.0f, gb = 0.0f;
    const int nchunk = (int)(((long long)n + SC - 1) / SC);
    for (int c = blockIdx.x; c < nchunk; c += gridDim.x) {
        const long long s0 = (long long)c * SC;
        const int ns = (int)min((long long)SC, n - s0);
        __syncthreads();
        {
            // thread: sample t / 4, four features (samples beyond n: zeros)
            const int s = t >> 2, f = 4 * (t & 3);
            const float4 v = s < ns ? *reinterpret_cast<const float4 *>(x + (s0 + s) * NI + f) : float4{0, 0, 0, 0};
            L.X[f][s] = v.x; L.X[f + 1][s] = v.y; L.X[f + 2][s] = v.z; L.X[f + 3][s] = v.w;
        }
        __syncthreads();
        float a[4][4];
        auto store = [&](float (*D)[SP]) {
#pragma unroll
            for (int b = 0; b < 4; ++b) row4(&D[tc + 16 * b][4 * tr]) = float4{a[b][0], a[b][1], a[b][2], a[b][3]};
        };
        auto layer = [&](float (*W)[NH], float (*V)[SP], const float *bias, int k, int ldw) {
            const float *w = &W[0][0];
#pragma unroll
            for (int b = 0; b < 4; ++b)
#pragma unroll
                for (int q = 0; q < 4; ++q) a[b][q] = bias[tc + 16 * b];
#pragma unroll 4
            for (int i = 0; i < k; ++i) {
                const float4 v = row4(&V[i][4 * tr]);
#pragma unroll
                for (int b = 0; b < 4; ++b) fma4(a[b], w[i * ldw + tc + 16 * b], v);
            }
#pragma unroll
            for (int b = 0; b < 4; ++b)
#pragma unroll
                for (int q = 0; q < 4; ++q) a[b][q] = fmaxf(a[b][q], 0.0f);
        };
        layer(L.W1, L.X, L.b1, NI, NH);
        store(L.H1);
        __syncthreads();
        layer(reinterpret_cast<float (*)[NH]>(&L.W2[0][0]), L.H1, L.b2, NH, SP);
        store(L.H2);
        __syncthreads();
        if (t < NO * SC) {
            const int o = t >> 6, s = t & 63;
            float z = L.b3[o];
#pragma unroll 8
            for (int j = 0; j < NH; ++j) z = fmaf(L.H2[j][s], L.W3[j * NO + o], z);
            L.z[o][s] = z;
        }
        __syncthreads();
        if (t < SC) {
            float z[NO], e[NO], se = 0.0f;
#pragma unroll
            for (int o = 0; o < NO; ++o) z[o] = L.z[o][t];
            const float zm = fmaxf(fmaxf(z[0], z[1]), z[2]);
#pragma unroll
            for (int o = 0; o < NO; ++o) { e[o] = expf(z[o] - zm); se += e[o]; }
#pragma unroll
            for (int o = 0; o < NO; ++o) e[o] = e[o] / se;
            if constexpr (GRAD) {
                const bool in = t < ns;
                const int ys = in ? y[s0 + t] : 0;
                const float w = in ? cw[ys] * inv_wsum : 0.0f;
                float py = 1.0f;
#pragma unroll
                for (int o = 0; o < NO; ++o) {
                    L.d3[o][t] = w * (e[o] - (o == ys ? 1.0f : 0.0f));
                    py = (o == ys) ? e[o] : py;
                }
                L.loss[t] = in ? -w * logf(fmaxf(py, 1e-30f)) : 0.0f;
            } else if (t < ns) {
#pragma unroll
                for (int o = 0; o < NO; ++o) prob[(s0 + t) * NO + o] = e[o];
            }
        }
        if constexpr (GRAD) {
            __syncthreads();
            // output layer's gradient (threads 0 .. 191: unit t / 3, class t % 3), its bias and the loss
            if (t < NH * NO) {
                const int j = t / NO, o = t % NO;
#pragma unroll 4
                for (int s = 0; s < SC; s += 4) g3 = dot4(g3, row4(&L.H2[j][s]), row4(&L.d3[o][s]));
            } else if (t < NH * NO + NO + 1) {
                const float *v = t < NH * NO + NO ? L.d3[t - NH * NO] : L.loss;
                for (int s = 0; s < SC; ++s) gb += v[s];
            }
            // delta of layer 2 in place of its activations
            float4 dv[NO];
#pragma unroll
            for (int o = 0; o < NO; ++o) dv[o] = row4(&L.d3[o][4 * tr]);
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const int j = tc + 16 * b;
                float acc[4] = {0, 0, 0, 0};
#pragma unroll
                for (int o = 0; o < NO; ++o) fma4(acc, L.W3[j * NO + o], dv[o]);
                const float4 hv = row4(&L.H2[j][4 * tr]);
                a[b][0] = hv.x > 0.0f ? acc[0] : 0.0f;
                a[b][1] = hv.y > 0.0f ? acc[1] : 0.0f;
                a[b][2] = hv.z > 0.0f ? acc[2] : 0.0f;
                a[b][3] = hv.w > 0.0f ? acc[3] : 0.0f;
            }
            __syncthreads();
            store(L.H2);
            __syncthreads();
            // delta of layer 1
#pragma unroll
            for (int b = 0; b < 4; ++b)
#pragma unroll
                for (int q = 0; q < 4; ++q) a[b][q] = 0.0f;
#pragma unroll 4
            for (int j = 0; j < NH; ++j) {
                const float4 v = row4(&L.H2[j][4 * tr]);
#pragma unroll
                for (int b = 0; b < 4; ++b) fma4(a[b], L.W2[tc + 16 * b][j], v);
            }
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const float4 hv = row4(&L.H1[tc + 16 * b][4 * tr]);
                a[b][0] = hv.x > 0.0f ? a[b][0] : 0.0f;
                a[b][1] = hv.y > 0.0f ? a[b][1] : 0.0f;
                a[b][2] = hv.z > 0.0f ? a[b][2] : 0.0f;
                a[b][3] = hv.w > 0.0f ? a[b][3] : 0.0f;
            }
            store(L.D1);
            __syncthreads();
            // gradients of the hidden layers: inputs tr + 16 q, units tc + 16 b, summed over samples
#pragma unroll 2
            for (int s = 0; s < SC; s += 4) {
                float4 hv[4], d2[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) { hv[q] = row4(&L.H1[tr + 16 * q][s]); d2[q] = row4(&L.H2[tc + 16 * q][s]); }
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int b = 0; b < 4; ++b) g2[q][b] = dot4(g2[q][b], hv[q], d2[b]);
                const float4 xv = row4(&L.X[tr][s]);
#pragma unroll
                for (int b = 0; b < 4; ++b) g1[b] = dot4(g1[b], xv, row4(&L.D1[tc + 16 * b][s]));
            }
            if (t < 2 * NH) {
                float *v = t < NH ? L.D1[t] : L.H2[t - NH];
                float acc = 0.0f;
                for (int s = 0; s < SC; s += 4) acc += (row4(v + s).x + row4(v + s).y) + (row4(v + s).z + row4(v + s).w);
                gb += acc;
            }
        }
    }
    if constexpr (GRAD) {
        float *P = part + (size_t)blockIdx.x * (NPAR + 1);
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            P[O_W1 + tr * NH + tc + 16 * b] = g1[b];
#pragma unroll
            for (int q = 0; q < 4; ++q) P[O_W2 + (tr + 16 * q) * NH + tc + 16 * b] = g2[q][b];
        }
        if (t < NH) P[O_B1 + t] = gb;
        else if (t < 2 * NH) P[O_B2 + t - NH] = gb;
        else if (t >= NH * NO && t < NH * NO + NO + 1) P[O_B3 + t - NH * NO] = gb;  // (the loss follows the parameters)
        if (t < NH * NO) P[O_W3 + t] = g3;
    }
}

// Sums of the workgroups' partial gradients, in workgroup order within four interleaved sequences;
// 64 parameters per workgroup.
__global__ __launch_bounds__(256) void k_mlp_reduce(int np, const float *__restrict__ part, float *__restrict__ grad) {
    __shared__ float s[4][64];
    const int l = threadIdx.x & 63, g = threadIdx.x >> 6, q = blockIdx.x * 64 + l;
    float acc = 0.0f;
    if (q <= NPAR)
#pragma unroll 8
        for (int b = g; b < np; b += 4) acc += part[(size_t)b * (NPAR + 1) + q];
    s[g][l] = acc;
    __syncthreads();
    if (g == 0 && q <= NPAR) grad[q] = (s[0][l] + s[1][l]) + (s[2][l] + s[3][l]);
}

// Adam (Kingma & Ba 2015) with bias correction.
__global__ __launch_bounds__(256) void k_mlp_adam(float *__restrict__ par, const float *__restrict__ grad,
                                                  float *__restrict__ m1, float *__restrict__ m2, float lr,
                                                  float c1, float c2) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= NPAR) return;
    const float g = grad[q];
    const float a = 0.9f * m1[q] + 0.1f * g;
    const float b = 0.999f * m2[q] + 0.001f * g * g;
    m1[q] = a;
    m2[q] = b;
    par[q] -= lr * (a / c1) / (sqrtf(b / c2) + 1e-8f);
}

// One device allocation for a gradient or a training run (grad: NPAR entries, then the loss).
struct Workspace {
    int n, np;
    float *par, *x, *grad, *part, *m1, *m2, *cw;
    int *y;
    char *base = nullptr;
    explicit Workspace(int n_) : n(n_), np((int)std::min<long long>(((long long)n_ + SC - 1) / SC, GRID)) {
        size_t at = 0;
        auto take = [&](size_t count) {
            const size_t o = at;
            at += (count * sizeof(float) + 255) / 256 * 256;
            return o;
        };
        const size_t o_par = take(NPAR), o_x = take((size_t)n * NI), o_grad = take(NPAR + 1),
                     o_part = take((size_t)np * (NPAR + 1)), o_m1 = take(NPAR), o_m2 = take(NPAR), o_cw = take(NO),
                     o_y = take(n);
        MLP_HIP(hipMalloc(&base, at));
        auto f = [&](size_t o) { return reinterpret_cast<float *>(base + o); };
        par = f(o_par); x = f(o_x); grad = f(o_grad); part = f(o_part); m1 = f(o_m1); m2 = f(o_m2); cw = f(o_cw);
        y = reinterpret_cast<int *>(base + o_y);
    }
    ~Workspace() { if (base) (void)hipFree(base); }
    Workspace(const Workspace &) = delete;
    Workspace &operator=(const Workspace &) = delete;
};

float weight_sum(int n, const int *y, const float *cw) {
    double s = 0.0;
    for (int i = 0; i < n; ++i) {
        if (y[i] < 0 || y[i] >= NO) throw std::invalid_argument("label out of range");
        s += cw ? cw[y[i]] : 1.0f;
    }
    if (!(s > 0.0)) throw std::invalid_argument("class weights sum to zero");
    return (float)(1.0 / s);
}

void upload(Workspace &w, const float *par, const float *x, const int *y, const float *cw) {
    MLP_HIP(hipMemcpy(w.par, par, NPAR * sizeof(float), hipMemcpyHostToDevice));
    MLP_HIP(hipMemcpy(w.x, x, (size_t)w.n * NI * sizeof(float), hipMemcpyHostToDevice));
    MLP_HIP(hipMemcpy(w.y, y, (size_t)w.n * sizeof(int), hipMemcpyHostToDevice));
    float ones[NO];
    for (float &o : ones) o = 1.0f;
    MLP_HIP(hipMemcpy(w.cw, cw ? cw : ones, NO * sizeof(float), hipMemcpyHostToDevice));
}

void grad_step(Workspace &w, float inv_wsum) {
    hipLaunchKernelGGL(k_mlp<true>, dim3((unsigned)w.np), dim3(256), 0, 0, w.par, w.n, w.x, w.y, w.cw, inv_wsum,
                       (float *)nullptr, w.part);
    hipLaunchKernelGGL(k_mlp_reduce, dim3((NPAR + 1 + 63) / 64), dim3(256), 0, 0, w.np, w.part, w.grad);
    MLP_HIP(hipGetLastError());
}

}  // namespace

// Inference buffers (parameters, features, probabilities) and a non-blocking stream (default
// priority) per device, made on first use and kept until the process ends: a forward pass per
// factorization allocates nothing after the first and does not wait for other streams' work (a
// solve running on the device meanwhile).
struct FwdBufs {
    float *par = nullptr, *x = nullptr, *prob = nullptr;
    size_t cap = 0;
    hipStream_t st = nullptr;
};

void mlp_forward(const float *par, int n, const float *x, float *prob) {
    if (n <= 0) return;
    static std::mutex mu;
    static std::map<int, FwdBufs> bufs;
    std::lock_guard<std::mutex> lock(mu);
    int dev = 0;
    MLP_HIP(hipGetDevice(&dev));
    FwdBufs &b = bufs[dev];
    if (!b.st) MLP_HIP(hipStreamCreateWithFlags(&b.st, hipStreamNonBlocking));
    if (!b.par) MLP_HIP(hipMalloc(&b.par, NPAR * sizeof(float)));
    if ((size_t)n > b.cap) {
        if (b.x) (void)hipFree(b.x);
        if (b.prob) (void)hipFree(b.prob);
        b.x = b.prob = nullptr;
        b.cap = 0;
        const size_t cap = std::max<size_t>((size_t)n, 4096);
        MLP_HIP(hipMalloc(&b.x, cap * NI * sizeof(float)));
        MLP_HIP(hipMalloc(&b.prob, cap * NO * sizeof(float)));
        b.cap = cap;
    }
    MLP_HIP(hipMemcpyAsync(b.par, par, NPAR * sizeof(float), hipMemcpyHostToDevice, b.st));
    MLP_HIP(hipMemcpyAsync(b.x, x, (size_t)n * NI * sizeof(float), hipMemcpyHostToDevice, b.st));
    const unsigned gs = (unsigned)std::min<long long>(((long long)n + SC - 1) / SC, GRID);
    hipLaunchKernelGGL(k_mlp<false>, dim3(gs), dim3(256), 0, b.st, b.par, n, b.x, (const int *)nullptr,
                       (const float *)nullptr, 0.0f, b.prob, (float *)nullptr);
    MLP_HIP(hipGetLastError());
    MLP_HIP(hipMemcpyAsync(prob, b.prob, (size_t)n * NO * sizeof(float), hipMemcpyDeviceToHost, b.st));
    MLP_HIP(hipStreamSynchronize(b.st));
}

void mlp_loss_grad(const float *par, int n, const float *x, const int *y, const float *cw, float *loss,
                   float *grad) {
    if (n <= 0) throw std::invalid_argument("no samples");
    const float iw = weight_sum(n, y, cw);
    Workspace w(n);
    upload(w, par, x, y, cw);
    grad_step(w, iw);
    float out[NPAR + 1];
    MLP_HIP(hipMemcpy(out, w.grad, sizeof(out), hipMemcpyDeviceToHost));
    std::copy(out, out + NPAR, grad);
    *loss = out[NPAR];
}

void mlp_train(float *par, int n, const float *x, const int *y, const float *cw, int epochs, float lr,
               float *final_loss) {
    if (n <= 0) throw std::invalid_argument("no samples");
    if (epochs < 0 || !(lr > 0.0f)) throw std::invalid_argument("epochs >= 0 and lr > 0 required");
    const float iw = weight_sum(n, y, cw);
    Workspace w(n);
    upload(w, par, x, y, cw);
    MLP_HIP(hipMemset(w.m1, 0, NPAR * sizeof(float)));
    MLP_HIP(hipMemset(w.m2, 0, NPAR * sizeof(float)));
    double c1 = 1.0, c2 = 1.0;
    for (int e = 0; e < epochs; ++e) {
        grad_step(w, iw);
        c1 *= 0.9;
        c2 *= 0.999;
        hipLaunchKernelGGL(k_mlp_adam, dim3((NPAR + 255) / 256), dim3(256), 0, 0, w.par, w.grad, w.m1,
                           w.m2, lr, (float)(1.0 - c1), (float)(1.0 - c2));
        MLP_HIP(hipGetLastError());
    }
    // loss of the final parameters
    grad_step(w, iw);
    MLP_HIP(hipMemcpy(par, w.par, NPAR * sizeof(float), hipMemcpyDeviceToHost));
    if (final_loss) MLP_HIP(hipMemcpy(final_loss, w.grad + NPAR, sizeof(float), hipMemcpyDeviceToHost));
}

}  // namespace rv
