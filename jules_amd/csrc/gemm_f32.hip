// gemm_f32.hip - fp32 fused GEMM + bias + activation, and the elementwise
// activations, for gfx950.
//
// Semantics follow the reference's tiled AVX-512 kernel
// (include/jules/Kernel/FusedKernels.h:378-458, bias epilogue :308-313):
// every output is ONE sequential fma chain over k = 0..K-1 starting from 0
// (the reference reloads the stored partial sum per K tile and keeps chaining,
// :401-406), followed by + bias[j] and the vector-path activation.  The fp32
// MFMAs compute that chain bit for bit (gemm_f32_tile.hpp), so the GEMM runs
// on them, with no split of K.  Against thread tiles of v_fma_f32: 2000 x 3072
// x 1024 305 -> 113 us, 512^3 12.3 -> 8.0 us with its operands cold.
#include "common.hpp"
#include "launch.hpp"

namespace jh {
namespace {

template <int ACT>
__global__ void activation_kernel(float* out, const float* __restrict__ in, int64_t n) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
        out[i] = activate<ACT>(in[i]);
}

// fusedGelu (reference FusedKernels.h:606-627): gelu_zmm on the full groups
// of 16 elements, and on the last partial group (the n % 16 elements from
// n & ~15 on) the scalar formula with tanhf, evaluated left to right as the
// reference's tail loop is compiled: x + (0.044715*x*x)*x is one fma.
__global__ void fused_gelu_kernel(float* out, const float* __restrict__ in, int64_t n) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    const int64_t nv = n & ~int64_t(15);
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        const float x = in[i];
        out[i] = i < nv ? gelu(x)
                        : 0.5f * x * (1.0f + tanhf(0.7978845608f * __builtin_fmaf(0.044715f * x * x, x, x)));
    }
}

}  // namespace

hipError_t launch_gemm_f32(int act, const float* A, const float* B, const float* bias, float* C,
                           int M, int N, int K, hipStream_t s) {
    const F32Gemm g = {false, false, A, K, B, N, C, N, M, N, K, F32_EPI_ACT, act, bias, nullptr, 0, 1.0f, 0.0f, nullptr};
    return launch_f32_gemm(g, 1, 0, nullptr, s, 0.0f);
}

hipError_t launch_activation(int act, float* out, const float* in, int64_t n, hipStream_t s) {
    if (n == 0) return hipSuccess;
    const int threads = 256;
    int64_t blocks = (n + threads - 1) / threads;
    if (blocks > 4096) blocks = 4096;
    if (act == JH_ACT_GELU) {
        hipLaunchKernelGGL(fused_gelu_kernel, dim3((unsigned)blocks), dim3(threads), 0, s, out, in, n);
        return hipGetLastError();
    }
    hipError_t e = hipSuccess;
    JH_DISPATCH_ACT(act, ACT, {
        hipLaunchKernelGGL(activation_kernel<ACT>, dim3((unsigned)blocks), dim3(threads), 0, s,
                           out, in, n);
        e = hipGetLastError();
    });
    return e;
}

}  // namespace jh
