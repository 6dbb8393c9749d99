// gemm_f32_kernel.hpp - the kernel of the fp32 MFMA GEMM tiles and its launch
// for one pair of operand orientations (gemm_f32_tile.hip and
// gemm_f32_tile_t.hip compile it for op(A) op(B) without and with transposes).
#pragma once

#include "gemm_f32_tile.hpp"
#include "gemm_tile.hpp"

namespace jh {

template <int MF_, int MT_, int NT_, int BK_, int PF_>
struct F32Cfg {
    static constexpr int MF = MF_, MT = MT_, NT = NT_, BK = BK_, PF = PF_;
    static constexpr int BM = 2 * MT * MF, BN = 2 * NT * MF;
};

// The epilogue g.epi over each(f), which calls f(m, n, sum, bias of column n),
// and read_each(load, f), which takes load(m, n) of every output of a thread before
// the first f(m, n, sum, loaded): one after the other, each load waited for the
// store before it (5935 x 1715 x 85 with beta 1 took 87 us, so 44).
// ACTS: with the activations (the transposed products only take "none").
template <bool ACTS, typename Each, typename ReadEach>
__device__ __forceinline__ void finish(const F32Gemm& g, Each&& each, ReadEach&& read_each) {
    if (g.epi == F32_EPI_MASK) {
        read_each([&](int m, int n) { return g.mask[(int64_t)m * g.ldm + n]; },
                  [&](int m, int n, float v, float a) { g.C[(int64_t)m * g.ldc + n] = a > 0.0f ? v : 0.0f; });
    } else if (g.epi == F32_EPI_ALPHA_BETA && g.beta == 0.0f) {
        // C is not read, so NaNs in an uninitialised one never propagate
        each([&](int m, int n, float v, float) { g.C[(int64_t)m * g.ldc + n] = g.alpha * v; });
    } else if (g.epi == F32_EPI_ALPHA_BETA) {
        read_each([&](int m, int n) { return g.C[(int64_t)m * g.ldc + n]; },
                  [&](int m, int n, float v, float c) { g.C[(int64_t)m * g.ldc + n] = g.alpha * v + g.beta * c; });
    } else if constexpr (ACTS) {
        JH_DISPATCH_ACT(g.act, ACT, each([&](int m, int n, float v, float b) {
                            if (g.bias) v = v + b;
                            g.C[(int64_t)m * g.ldc + n] = activate<ACT>(v);
                        }));
    } else {
        each([&](int m, int n, float v, float) {
            float* c = g.colsum && m == g.M - 1 ? g.colsum + n : g.C + (int64_t)m * g.ldc + n;
            *c = v;
        });
    }
}

template <class CF, bool TA, bool TB, int V, bool FOLD>
__global__ __launch_bounds__(256, 2) void gemm_f32_tile_kernel(F32Gemm g, int kc, int chunk, float* __restrict__ part) {
    using T = F32Tile<CF::MF, CF::MT, CF::NT, CF::BK, CF::PF, TA, TB, V, FOLD>;
    constexpr bool ACTS = !TA && !TB;
    __shared__ __attribute__((aligned(16))) float sm[2 * T::STAGE];
    const TileCoord t = tile_coord<8>((g.M + (T::BM - 1)) / T::BM, (g.N + (T::BN - 1)) / T::BN);
    const int m0 = t.tm * T::BM, n0 = t.tn * T::BN, kb = t.z * kc;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int mw = m0 + (wave >> 1) * CF::MT * CF::MF, nw = n0 + (wave & 1) * CF::NT * CF::MF + lane % CF::MF;
    // the bias is in registers before the sums are (loaded after them, it costs
    // a small product a memory latency)
    float bias[CF::NT];
#pragma unroll
    for (int j = 0; j < CF::NT; ++j)
        bias[j] = ACTS && g.bias ? g.bias[min(nw + j * CF::MF, g.N - 1)] : 0.0f;

    typename T::Mf::Acc acc[CF::MT][CF::NT];
    T::run(g.A, g.lda, g.B, g.ldb, m0, g.M - (g.colsum ? 1 : 0), n0, g.N, kb, min(g.K, kb + kc), chunk,
           g.colsum != nullptr, sm, acc);

    auto each = [&](auto&& f) {
#pragma unroll
        for (int j = 0; j < CF::NT; ++j) {
            const int n = nw + j * CF::MF;
            if (n >= g.N) continue;
#pragma unroll
            for (int i = 0; i < CF::MT; ++i)
#pragma unroll
                for (int e = 0; e < T::Mf::NR; ++e) {
                    const int m = mw + i * CF::MF + T::Mf::row(lane, e);
                    if (m < g.M) f(m, n, acc[i][j][e], bias[j]);
                }
        }
    };
    if (part) {
        float* p = part + (int64_t)t.z * g.M * g.N;
        each([&](int m, int n, float v, float) { p[(int64_t)m * g.N + n] = v; });
    } else {
        finish<ACTS>(g, each, [&](auto&& load, auto&& f) {
            // All 64 outputs of a 128 x 128 tile at once take 232 registers, which
            // leaves two workgroups on a CU, not three (5936 x 1716 x 96, beta 0 too,
            // 34 -> 45 us): there an accumulator at a time, or with A transposed,
            // where that still costs the tile 10 %, one by one.
            if constexpr (CF::MT * CF::NT * T::Mf::NR > 32 && TA) {
                each([&](int m, int n, float v, float) { f(m, n, v, load(m, n)); });
            } else if constexpr (CF::MT * CF::NT * T::Mf::NR > 32) {
#pragma unroll
                for (int j = 0; j < CF::NT; ++j) {
                    const int n = nw + j * CF::MF;
                    if (n >= g.N) continue;
#pragma unroll
                    for (int i = 0; i < CF::MT; ++i) {
                        const int mi = mw + i * CF::MF;
                        float x[T::Mf::NR];
#pragma unroll
                        for (int e = 0; e < T::Mf::NR; ++e)
                            x[e] = load(min(mi + T::Mf::row(lane, e), g.M - 1), n);  // past the end: not used
#pragma unroll
                        for (int e = 0; e < T::Mf::NR; ++e) {
                            const int m = mi + T::Mf::row(lane, e);
                            if (m < g.M) f(m, n, acc[i][j][e], x[e]);
                        }
                    }
                }
            } else {
                float x[CF::NT][CF::MT][T::Mf::NR];
                // rows and columns past the end as the last: what they load is not used
                const auto row = [&](int i, int e) { return mw + i * CF::MF + T::Mf::row(lane, e); };
#pragma unroll
                for (int j = 0; j < CF::NT; ++j)
#pragma unroll
                    for (int i = 0; i < CF::MT; ++i)
#pragma unroll
                        for (int e = 0; e < T::Mf::NR; ++e)
                            x[j][i][e] = load(min(row(i, e), g.M - 1), min(nw + j * CF::MF, g.N - 1));
#pragma unroll
                for (int j = 0; j < CF::NT; ++j)
#pragma unroll
                    for (int i = 0; i < CF::MT; ++i)
#pragma unroll
                        for (int e = 0; e < T::Mf::NR; ++e)
                            if (row(i, e) < g.M && nw + j * CF::MF < g.N)
                                f(row(i, e), nw + j * CF::MF, acc[i][j][e], x[j][i][e]);
            }
        });
    }
}

using F32Cfg0 = F32Cfg<16, 1, 1, 64, 1>;
using F32Cfg1 = F32Cfg<16, 2, 2, 32, 2>;
using F32Cfg2 = F32Cfg<16, 2, 4, 16, 1>;
using F32Cfg3 = F32Cfg<32, 2, 2, 16, 1>;
using F32Cfg4 = F32Cfg<16, 1, 1, 128, 1>;

template <bool TA, bool TB>
void launch_f32_tile(int plan, int v, const F32Gemm& g, int splits, int kc, int chunk, float* part, hipStream_t s) {
    using yes = std::integral_constant<bool, true>;
    using no = std::integral_constant<bool, false>;
    auto go = [&](auto cfg, auto vec, auto fold) {
        using CF = decltype(cfg);
        const int64_t wg =
            (((int64_t)g.M + CF::BM - 1) / CF::BM) * (((int64_t)g.N + CF::BN - 1) / CF::BN) * splits;
        hipLaunchKernelGGL((gemm_f32_tile_kernel<CF, TA, TB, decltype(vec)::value, decltype(fold)::value>), dim3((unsigned)wg), dim3(256), 0,
                           s, g, kc, chunk, part);
    };
    auto pick = [&](auto vec) {
        switch (plan) {
        case 0: chunk ? go(F32Cfg0{}, vec, yes{}) : go(F32Cfg0{}, vec, no{}); break;
        case 1: go(F32Cfg1{}, vec, no{}); break;
        case 2: go(F32Cfg2{}, vec, no{}); break;
        case 3:
            // a transposed B's fragments spill at 128 x 128 (64 x 128 is within 4 %)
            if constexpr (TB) go(F32Cfg2{}, vec, no{});
            else go(F32Cfg3{}, vec, no{});
            break;
        default: chunk ? go(F32Cfg4{}, vec, yes{}) : go(F32Cfg4{}, vec, no{}); break;
        }
    };
    if (v == 4) pick(std::integral_constant<int, 4>{});
    else if (v == 1) pick(std::integral_constant<int, 1>{});
    else if (chunk) go(F32Cfg0{}, std::integral_constant<int, 0>{}, yes{});
    else go(F32Cfg0{}, std::integral_constant<int, 0>{}, no{});
}

// gemm_f32_tile_t.hip: at least one of ta, tb
void launch_f32_tile_trans(int plan, int v, const F32Gemm& g, int splits, int kc, int chunk, float* part, hipStream_t s);

}  // namespace jh
