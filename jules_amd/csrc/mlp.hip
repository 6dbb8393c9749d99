// mlp.hip - 2-layer MLP forward + softmax cross entropy + backward on gfx950.
//
// Reference: interleavedMLPForwardBackward (include/jules/Kernel/
// InterleavedAutodiff.h:55-441):
//   h = X W1 + b1, a = relu(h)                               :144-166
//   o = a W2 + b2 -> output                                  :168-176
//   p = softmax(o) per row, loss = sum_i -log(p[t_i] + 1e-10) / M,
//   dO = (p - onehot(t)) / M                                 :178-197
//   dW2 = a^T dO, db2 = colsum(dO)                           :207-221
//   dA = dO W2^T, dH = dA * (h > 0)                          :223-247
//   dW1 = X^T dH, db1 = colsum(dH), dX = dH W1^T             :249-267
// The reference runs this tile by tile on the CPU so that h and a stay in
// cache between the forward and the backward of a tile.  Here the five
// products are whole-matrix fp32 MFMA GEMMs and the intermediates (a, dO,
// dH) go to a caller workspace in HBM: at the shapes where the GPU pays off
// they are a few per cent of the GEMM traffic, and whole-matrix GEMMs keep
// the MFMA pipes full where tile-sized ones would not.
//
// relu'(h) is read from a: a > 0 exactly when h > 0, so h is not stored.
// The loss and dO come from the fused cross-entropy row kernel (rowops.hip),
// which computes the same formula.  db1/db2 are column sums in a fixed order
// (row chunks, then the chunks in order), so every result is deterministic.
//
// The products run on the fp32 MFMA tiles of gemm_f32_tile.hip.
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "launch.hpp"

namespace jh {
namespace {

// C = beta * C (alpha * op(A) op(B) vanishes: K = 0 or alpha = 0); beta = 0
// writes zeros without reading C, as BLAS does
__global__ void scale_c_kernel(float* __restrict__ C, int ldc, int M, int N, float beta) {
    const int64_t total = (int64_t)M * N, stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += stride) {
        const int m = (int)(e / N), n = (int)(e - (int64_t)m * N);
        float* c = C + (int64_t)m * ldc + n;
        *c = beta == 0.0f ? 0.0f : beta * *c;
    }
}

// Column sums in a fixed order: partial[s][n] sums rows [s*R, (s+1)*R) in
// row order, then out[n] sums the partials in s order.
__global__ void colsum_partial_kernel(const float* __restrict__ X, int M, int N, int ld, int R,
                                      float* __restrict__ part) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    const int s = blockIdx.y;
    if (n >= N) return;
    const int r0 = s * R, r1 = min(M, r0 + R);
    float acc = 0.0f;
    int m = r0;
    // 8 loads in flight, added in row order
    for (; m + 8 <= r1; m += 8) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = X[(int64_t)(m + u) * ld + n];
#pragma unroll
        for (int u = 0; u < 8; ++u) acc += v[u];
    }
    for (; m < r1; ++m) acc += X[(int64_t)m * ld + n];
    part[(int64_t)s * N + n] = acc;
}

__global__ void colsum_final_kernel(const float* __restrict__ part, int S, int N,
                                    float* __restrict__ out) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= N) return;
    float acc = part[n];
    for (int s = 1; s < S; ++s) acc += part[(int64_t)s * N + n];
    out[n] = acc;
}

__global__ void fill_kernel(float* __restrict__ p, int64_t n, float v) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) p[i] = v;
}

// K ranges of a product, each summed by itself: one with fewer than 128 output
// tiles of 128 x 128 sums K in as many ranges (of at least 64) as would make
// about 256 of them.  They say in which order the products are summed; whether
// a range gets workgroups of its own is launch_f32_gemm's choice, and the
// workspace holds their partial sums in case it does.
constexpr int BM = 128, BN = 128, BK = 16;
struct KPlan {
    int S;   // ranges
    int kc;  // K elements per range, a multiple of BK
};

KPlan kplan(int M, int N, int K) {
    // 64-bit: M, N, K may be anywhere up to INT_MAX
    const int64_t tiles = ((int64_t)M + BM - 1) / BM * (((int64_t)N + BN - 1) / BN);
    const int max_s = K / (4 * BK);
    if (tiles <= 0 || tiles >= 128 || max_s < 2) return {1, K};
    int S = (int)((256 + tiles - 1) / tiles);
    if (S > max_s) S = max_s;
    const int64_t kc = (((int64_t)K + S - 1) / S + BK - 1) / BK * BK;
    return {(int)(((int64_t)K + kc - 1) / kc), (int)kc};
}

size_t kplan_floats(int M, int N, int K) {
    const KPlan p = kplan(M, N, K);
    return p.S > 1 ? (size_t)p.S * M * N : 0;
}

// A training step's seven launches are as many as the host enqueues in its time:
// with an eighth the step of 64 rows took 36.9 us, not 34.4, though its first
// product was 2 us shorter.
constexpr float kStepLaunchUs = 5.0f;

hipError_t gemm(F32Gemm g, float* part, hipStream_t s, float launch_us = kStepLaunchUs) {
    const KPlan p = kplan(g.M, g.N, g.K);
    return launch_f32_gemm(g, p.S, p.kc, part, s, launch_us);
}
// X W + bias, with or without ReLU
F32Gemm layer(const float* X, const float* W, const float* bias, int act, float* Y, int M, int N, int K) {
    return {false, false, X, K, W, N, Y, N, M, N, K, F32_EPI_ACT, act, bias, nullptr, 0, 1.0f, 0.0f, nullptr};
}

constexpr int COLSUM_ROWS = 256;  // rows per partial column sum
constexpr int COLSUM_MAX_CHUNKS = 64;

int colsum_chunks(int M, int* rows) {
    int S = (M + COLSUM_ROWS - 1) / COLSUM_ROWS;
    if (S > COLSUM_MAX_CHUNKS) S = COLSUM_MAX_CHUNKS;
    if (S < 1) S = 1;
    *rows = (M + S - 1) / S;
    return S;
}

// dW = A^T G and db = colsum(G), A [M,Ka], G [M,N].  Up to COLSUM_ROWS rows the
// column sum is an extra row of ones in A^T, summed as the product is (a chain
// over the rows, or over each range of them); more rows are summed in chunks by
// kernels of their own.
hipError_t weight_grad(const float* A, int Ka, const float* G, int M, int N, float* dW, float* db,
                       float* colsum_part, float* part, hipStream_t s) {
    const bool fold = M <= COLSUM_ROWS;
    F32Gemm g = {true, false, A, Ka, G, N, dW, N, Ka + fold, N, M, F32_EPI_ACT, JH_ACT_NONE, nullptr, nullptr, 0,
                 1.0f, 0.0f, fold ? db : nullptr};
    const KPlan p = kplan(Ka, N, M);
    const hipError_t e = launch_f32_gemm(g, p.S, p.kc, fold ? nullptr : part, s, kStepLaunchUs);
    if (fold || e != hipSuccess) return e;
    int R;
    const int S = colsum_chunks(M, &R);
    hipLaunchKernelGGL(colsum_partial_kernel, dim3((N + 255) / 256, S), dim3(256), 0, s, G, M, N, N, R, colsum_part);
    hipLaunchKernelGGL(colsum_final_kernel, dim3((N + 255) / 256), dim3(256), 0, s, colsum_part, S, N, db);
    return hipGetLastError();
}

hipError_t fill(float* p, int64_t n, float v, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    int64_t b = (n + 255) / 256;
    if (b > 4096) b = 4096;
    hipLaunchKernelGGL(fill_kernel, dim3((unsigned)b), dim3(256), 0, s, p, n, v);
    return hipGetLastError();
}

size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

}  // namespace

// workspace: a [M,N1], dH [M,N1], dO [M,N2], per-row losses [M], column-sum
// partials [chunks, max(N1,N2)], each 256-byte aligned
size_t mlp_workspace_size(int M, int K1, int N1, int N2) {
    (void)K1;
    int R;
    const int S = colsum_chunks(M, &R);
    const size_t mn1 = (size_t)M * N1 * sizeof(float), mn2 = (size_t)M * N2 * sizeof(float);
    // split-K partials of the five products (only skinny ones split)
    size_t kp = kplan_floats(M, N1, K1);
    kp = std::max(kp, kplan_floats(M, N2, N1));
    kp = std::max(kp, kplan_floats(N1, N2, M));
    kp = std::max(kp, kplan_floats(M, N1, N2));
    kp = std::max(kp, kplan_floats(K1, N1, M));
    kp = std::max(kp, kplan_floats(M, K1, N1));
    return 2 * align256(mn1) + align256(mn2) + align256((size_t)M * sizeof(float)) +
           align256((size_t)S * (N1 > N2 ? N1 : N2) * sizeof(float)) + align256(kp * sizeof(float));
}

// fusedMLPForward (reference FusedKernels.h:659-760): output = relu(X W1 +
// b1) W2 + b2, the forward half of the step below.  workspace: the hidden
// activations [M,N1], then split-K partials
size_t mlp_forward_workspace_size(int M, int K1, int N1, int N2) {
    (void)K1;
    const size_t kp = std::max(kplan_floats(M, N1, K1), kplan_floats(M, N2, N1));
    return align256((size_t)M * N1 * sizeof(float)) + align256(kp * sizeof(float));
}

hipError_t launch_mlp_forward(const float* X, const float* W1, const float* b1, const float* W2,
                              const float* b2, float* output, int M, int K1, int N1, int N2,
                              void* ws, hipStream_t s) {
    if (M == 0) return hipSuccess;
    float* act = static_cast<float*>(ws);
    float* kpart = reinterpret_cast<float*>(static_cast<char*>(ws) +
                                            align256((size_t)M * N1 * sizeof(float)));
    const hipError_t e = gemm(layer(X, W1, b1, JH_ACT_RELU, act, M, N1, K1), kpart, s);
    if (e != hipSuccess) return e;
    return gemm(layer(act, W2, b2, JH_ACT_NONE, output, M, N2, N1), kpart, s);
}

hipError_t launch_mlp_forward_backward(const float* X, const float* W1, const float* b1,
                                       const float* W2, const float* b2, const int32_t* targets,
                                       float* output, float* dW1, float* db1, float* dW2, float* db2,
                                       float* dX, float* loss, int M, int K1, int N1, int N2,
                                       void* ws, hipStream_t s) {
    if (M == 0) {
        // no rows: zero gradients, loss 0/0 (the reference divides its
        // empty sum by M)
        hipError_t e = fill(dW1, (int64_t)K1 * N1, 0.0f, s);
        if (e == hipSuccess) e = fill(db1, N1, 0.0f, s);
        if (e == hipSuccess) e = fill(dW2, (int64_t)N1 * N2, 0.0f, s);
        if (e == hipSuccess) e = fill(db2, N2, 0.0f, s);
        if (e == hipSuccess) e = fill(loss, 1, __builtin_nanf(""), s);
        return e;
    }
    char* w = static_cast<char*>(ws);
    const size_t mn1 = align256((size_t)M * N1 * sizeof(float));
    const size_t mn2 = align256((size_t)M * N2 * sizeof(float));
    float* act = reinterpret_cast<float*>(w);
    float* dH = reinterpret_cast<float*>(w + mn1);
    float* dO = reinterpret_cast<float*>(w + 2 * mn1);
    float* row_loss = reinterpret_cast<float*>(w + 2 * mn1 + mn2);
    float* part = reinterpret_cast<float*>(w + 2 * mn1 + mn2 + align256((size_t)M * sizeof(float)));
    int R;
    const int S = colsum_chunks(M, &R);
    float* kpart = reinterpret_cast<float*>(reinterpret_cast<char*>(part) +
                                            align256((size_t)S * (N1 > N2 ? N1 : N2) * sizeof(float)));

    hipError_t e;
    // forward
    if ((e = gemm(layer(X, W1, b1, JH_ACT_RELU, act, M, N1, K1), kpart, s))) return e;
    if ((e = gemm(layer(act, W2, b2, JH_ACT_NONE, output, M, N2, N1), kpart, s))) return e;
    // loss and dO
    if ((e = launch_cross_entropy(output, targets, dO, loss, row_loss, M, N2, s))) return e;
    // layer 2 gradients
    if ((e = weight_grad(act, N1, dO, M, N2, dW2, db2, part, kpart, s))) return e;
    // dH = (dO W2^T) * (a > 0)
    const F32Gemm dh = {false, true, dO, N2, W2, N2, dH, N1, M, N1, N2, F32_EPI_MASK, JH_ACT_NONE, nullptr, act, N1,
                        1.0f, 0.0f, nullptr};
    if ((e = gemm(dh, kpart, s))) return e;
    // layer 1 gradients
    if ((e = weight_grad(X, K1, dH, M, N1, dW1, db1, part, kpart, s))) return e;
    if (!dX) return hipSuccess;
    const F32Gemm dx = {false, true, dH, N1, W1, N1, dX, K1, M, K1, N1, F32_EPI_ACT, JH_ACT_NONE, nullptr, nullptr, 0,
                        1.0f, 0.0f, nullptr};
    return gemm(dx, kpart, s);
}

// blasMatmul / cblas_sgemm (reference FusedKernels.h:633-644): the MFMA GEMM
// above with the sgemm epilogue.  Skinny products split K into a per-stream
// library buffer (the entry point has no workspace argument).
hipError_t launch_sgemm(bool transA, bool transB, int M, int N, int K, float alpha, const float* A,
                        int lda, const float* B, int ldb, float beta, float* C, int ldc,
                        hipStream_t s) {
    if (M == 0 || N == 0) return hipSuccess;
    if (K == 0 || alpha == 0.0f) {
        int64_t b = ((int64_t)M * N + 255) / 256;
        if (b > 4096) b = 4096;
        hipLaunchKernelGGL(scale_c_kernel, dim3((unsigned)b), dim3(256), 0, s, C, ldc, M, N, beta);
        return hipGetLastError();
    }
    float* part = nullptr;
    WorkspaceLock lock;
    const size_t pf = kplan_floats(M, N, K);
    if (pf) {
        void* ws = nullptr;
        const hipError_t e = stream_workspace(pf * sizeof(float), s, &ws, &lock);
        if (e != hipSuccess) return e;
        part = static_cast<float*>(ws);
    }
    return gemm({transA, transB, A, lda, B, ldb, C, ldc, M, N, K, F32_EPI_ALPHA_BETA, JH_ACT_NONE, nullptr, nullptr, 0,
                 alpha, beta, nullptr},
                part, s, 1.0f);
}

}  // namespace jh
