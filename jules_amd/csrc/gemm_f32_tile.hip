// gemm_f32_tile.hip - the launch of the fp32 MFMA GEMM (gemm_f32_tile.hpp): the
// fused GEMM of gemm_f32.hip, the MLP products and sgemm of mlp.hip.
#include <algorithm>

#include "gemm_f32_kernel.hpp"

namespace jh {
namespace {

// C = epilogue(sum over z of part[z], in z order)
__global__ __launch_bounds__(256) void gemm_f32_reduce_kernel(F32Gemm g, int S, const float* __restrict__ part) {
    const int64_t total = (int64_t)g.M * g.N, stride = (int64_t)gridDim.x * 256;
    const auto sums = [&](auto&& f) {
        for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < total; e += stride) {
            float v = part[e];
#pragma unroll 4
            for (int z = 1; z < S; ++z) v += part[(int64_t)z * total + e];
            const int m = (int)(e / g.N);
            f(m, (int)(e - (int64_t)m * g.N), v);
        }
    };
    finish<true>(
        g, [&](auto&& f) { sums([&](int m, int n, float v) { f(m, n, v, g.bias ? g.bias[n] : 0.0f); }); },
        [&](auto&& load, auto&& f) { sums([&](int m, int n, float v) { f(m, n, v, load(m, n)); }); });
}

// The tiles, and what they cost: n = ceil(workgroups / 256) tiles on a CU take
// n (k * per_k + round) us, one alone k * alone + round (its own latencies
// uncovered).  Measured at 4096^3, 2000 x 3072 x 1024, 1024^3 and 64 x 512 x
// 2048: per output the larger tiles are up to 1.4 times as fast (5.5 ns per k
// and 1024 outputs at 32 x 32, 4.0 at 128 x 128), the smaller ones fill the
// chip and split the fma chain's latency over more waves.
struct F32Plan {
    int bm, bn;
    float per_k, alone, round;
};
constexpr F32Plan kF32Plans[4] = {{32, 32, 0.0053f, 0.0062f, 1.0f},
                                  {64, 64, 0.0175f, 0.024f, 1.1f},
                                  {64, 128, 0.034f, 0.042f, 1.4f},
                                  {128, 128, 0.065f, 0.075f, 3.0f}};

int f32_plan(int M, int N, int kc, int splits, float* us_out) {
    int best = 0;
    float best_us = 0.0f;
    for (int c = 0; c < 4; ++c) {
        const F32Plan& p = kF32Plans[c];
        const int64_t wg = (((int64_t)M + p.bm - 1) / p.bm) * (((int64_t)N + p.bn - 1) / p.bn) * splits;
        const float n = (float)((wg + 255) / 256);
        const float us = n > 1.0f ? n * (kc * p.per_k + p.round) : kc * p.alone + p.round;
        if (c == 0 || us < best_us) {
            best_us = us;
            best = c;
        }
    }
    *us_out = best_us;
    // 32 x 32 tiles alone on their CUs: half as many barriers for a long chain
    // (64 x 512 x 2048 17.7 -> 15.9 us); with neighbours the larger LDS costs more
    if (best == 0 && kc >= 256 && ((int64_t)M + 31) / 32 * (((int64_t)N + 31) / 32) * splits <= 256) best = 4;
    return best;
}

struct F32Dims {
    int bm, bn, bk;
};
template <class CF>
constexpr F32Dims f32_dims() {
    return {CF::BM, CF::BN, CF::BK};
}
constexpr F32Dims kF32Dims[5] = {f32_dims<F32Cfg0>(), f32_dims<F32Cfg1>(), f32_dims<F32Cfg2>(),
                                 f32_dims<F32Cfg3>(), f32_dims<F32Cfg4>()};

// Whether every byte offset that the plan's tile forms (F32Slice::Src) is below
// 2^32: to each k of a slice, those past K among them, where k is the outer
// dimension in memory, and to each row that exists where it is not.
bool f32_fits(const F32Gemm& g, int plan) {
    const F32Dims& t = kF32Dims[g.tb && plan == 3 ? 2 : plan];  // as launch_f32_tile
    const auto span = [&](bool k_outer, int x, int rows, int64_t ld) {
        const int64_t xs = std::min(x, rows);
        return 4 * (k_outer ? (t.bk - 1) * ld + xs : (xs - 1) * ld + t.bk);
    };
    return std::max(span(g.ta, t.bm, g.M, g.lda), span(!g.tb, t.bn, g.N, g.ldb)) <= int64_t(1) << 32;
}

// One half of g's columns or, where there are more of them, its rows, whole
// 128 x 128 tiles in the first.
F32Gemm f32_half(F32Gemm g, bool second) {
    const bool cols = g.N >= g.M;
    const int at = (cols ? g.N : g.M) / 2 & ~127;
    if (!second) {
        (cols ? g.N : g.M) = at;
        if (!cols) g.colsum = nullptr;  // the last row of the second
        return g;
    }
    (cols ? g.N : g.M) -= at;
    if (cols) {
        g.B += g.tb ? at * g.ldb : at;
        if (g.bias) g.bias += at;
        if (g.colsum) g.colsum += at;
    } else {
        g.A += g.ta ? at : at * g.lda;
    }
    g.C += cols ? at : at * g.ldc;
    if (g.mask) g.mask += cols ? at : at * g.ldm;
    return g;
}

}  // namespace

// What 32 x 32 tiles that fold a long K's ranges take: its chain, one piece of k
// after the other, fitted to 1500 products with K 256-8192 in each orientation
// (within 0.5 to 1.5 us).  An operand whose k is outermost in memory and whose
// rows are no whole 16-byte pieces is loaded float by float.
static float f32_fold_us(const F32Gemm& g, bool vec) {
    const int64_t wg = (((int64_t)g.M + 31) / 32) * (((int64_t)g.N + 31) / 32);
    const float n = (float)((wg + 255) / 256);
    const float per_k = !g.ta && g.tb ? 0.0110f : vec || g.tb ? 0.0088f : g.ta ? 0.0133f : 0.0100f;
    return 4.0f + g.K * per_k * (n > 1.0f ? 0.7f * n : 1.0f);
}

hipError_t launch_f32_gemm(const F32Gemm& g, int splits, int kc, float* part, hipStream_t s, float launch_us) {
    if (g.M == 0 || g.N == 0) return hipSuccess;
    int chunk = 0, plan;
    float us;
    // whole 16-byte pieces of the operands whose k is the outer dimension
    const bool vec = (!g.ta || (g.M - (g.colsum ? 1 : 0)) % 4 == 0) && (g.tb || g.N % 4 == 0);
    if (splits > 1) {
        // The same sums in the same order in one launch, 32 x 32 tiles that fold
        // a range at a time, unless spreading the ranges over workgroups pays
        // for its reduction (825 x 74 x 2667, A transposed: 40 us folded, 23 in
        // two launches) and for what the caller says one launch more costs it.
        plan = f32_plan(g.M, g.N, kc, splits, &us);
        us += 4.5f + 0.07f * splits + 2.4e-6f * splits * g.M * g.N + launch_us;
        if (!part || f32_fold_us(g, vec) < us) {
            const int64_t wg = ((int64_t)g.M + 31) / 32 * (((int64_t)g.N + 31) / 32);
            chunk = kc;
            splits = 1;
            plan = wg <= 256 && g.K >= 256 ? 4 : 0;
        }
    }
    if (splits <= 1) {
        kc = g.K;
        part = nullptr;
        if (!chunk) plan = f32_plan(g.M, g.N, kc, 1, &us);
    }
    // a tile whose offsets pass 32 bits gives way to 32 x 32, then to 64-bit ones
    if (!f32_fits(g, plan)) plan = 0;
    const int v = !f32_fits(g, plan) ? 0 : vec ? 4 : 1;
    // the runtime takes fewer than 2^32 threads a launch
    const F32Dims& t = kF32Dims[g.tb && plan == 3 ? 2 : plan];  // as launch_f32_tile
    if (splits <= 1 && (((int64_t)g.M + t.bm - 1) / t.bm) * (((int64_t)g.N + t.bn - 1) / t.bn) >= int64_t(1) << 24) {
        const hipError_t e = launch_f32_gemm(f32_half(g, false), 1, 0, nullptr, s, 0.0f);
        return e != hipSuccess ? e : launch_f32_gemm(f32_half(g, true), 1, 0, nullptr, s, 0.0f);
    }
    if (g.ta || g.tb) launch_f32_tile_trans(plan, v, g, splits, kc, chunk, part, s);
    else launch_f32_tile<false, false>(plan, v, g, splits, kc, chunk, part, s);
    if (part) {
        int64_t b = ((int64_t)g.M * g.N + 255) / 256;
        if (b > 2048) b = 2048;
        hipLaunchKernelGGL(gemm_f32_reduce_kernel, dim3((unsigned)b), dim3(256), 0, s, g, splits, part);
    }
    return hipGetLastError();
}

}  // namespace jh
