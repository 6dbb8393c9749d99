// tiles.hpp - the gfx950 GEMM tile table of libjules_hip (internal).
//
// The table jules_hip_gemm_tile and jules::kernel::TilePlanner
// (kernel_shims.cpp) plan with (the reference's planner, TilePlanner.h:74-136,
// sizes tiles for the CPU caches instead).  It classifies shapes; within a
// class the launchers (gemm_f32_tile.hip, gemm_bf16.hip) pick the workgroup
// tile by their own measured costs.
//
// fp32 (the bit-exact fma-chain GEMM): every output is the same sequential fma
// chain over k whatever the entry, so the choice never changes bits.
//   F32_ROWS1 / F32_ROWS2: outputs so few that 4 or 8 rows x 64 columns over
//     all of K is a workgroup's share (K <= kF32RowsMaxK).
//   F32_T32 / F32_T64: 32x32 and 64x64 output tiles in K slices of 32.
// bf16 (MFMA): BF16_DMA, 256x256 output tiles of 4 waves over 32-deep K slices
// by LDS DMA, can run whole tiles only; BF16_REG stands for every other shape.
// Which kernel and tile a launch takes is the cost model of gemm_bf16.hip.
#pragma once

#include <stdint.h>

namespace jh {

enum GemmVariant {
    GV_F32_ROWS1 = 0,
    GV_F32_ROWS2 = 1,
    GV_F32_T32 = 2,
    GV_F32_T64 = 3,
    GV_BF16_DMA = 4,
    GV_BF16_REG = 5,
    GV_COUNT = 6
};

struct GemmTile {
    int variant;
    int tile_m;
    int tile_n;
    int tile_k;
};

constexpr int kF32RowsWaves = 4;     // waves of a rows entry
constexpr int kF32RowsMaxK = 2048;   // longest K of a rows entry
constexpr int kF32SliceK = 32;       // K slice of the 32x32 and 64x64 entries
constexpr int kBf16Tile = 256;       // bf16 output tile (both variants)
constexpr int kBf16DmaK = 32;        // k per LDS-DMA stage
constexpr int kBf16RegK = 64;        // k per register-staged slice

inline bool f32_variant_valid(int v, int K) {
    if (v == GV_F32_ROWS1 || v == GV_F32_ROWS2) return K <= kF32RowsMaxK;
    return v == GV_F32_T32 || v == GV_F32_T64;
}

inline GemmTile f32_variant_tile(int v, int K) {
    switch (v) {
    case GV_F32_ROWS1: return {v, kF32RowsWaves, 64, (K + 3) & ~3};
    case GV_F32_ROWS2: return {v, 2 * kF32RowsWaves, 64, (K + 3) & ~3};
    case GV_F32_T32: return {v, 32, 32, kF32SliceK};
    default: return {GV_F32_T64, 64, 64, kF32SliceK};
    }
}

// The entry of an fp32 shape.  Up to 1M outputs (and K <= kF32RowsMaxK): rows,
// 2 per wave, or 1 when 2 would leave fewer than 1024 waves.  Larger: 64x64
// tiles once there are at least 512 of them (two per CU), else 32x32.
inline GemmTile f32_gemm_tile(int M, int N, int K) {
    if ((int64_t)M * N <= (int64_t(1) << 20) && K <= kF32RowsMaxK) {
        const bool one = (((int64_t)N + 63) / 64) * (((int64_t)M + 1) / 2) < 1024;
        return f32_variant_tile(one ? GV_F32_ROWS1 : GV_F32_ROWS2, K);
    }
    const int64_t tiles64 = (((int64_t)M + 63) / 64) * (((int64_t)N + 63) / 64);
    return f32_variant_tile(tiles64 >= 512 ? GV_F32_T64 : GV_F32_T32, K);
}

// LDS DMA over whole tiles can run when M and N are multiples of the 256 tile
// and K of the 32-deep stage.
inline GemmTile bf16_gemm_tile(int M, int N, int K) {
    const bool full = M % kBf16Tile == 0 && N % kBf16Tile == 0 && K % kBf16DmaK == 0 && K > 0;
    return full ? GemmTile{GV_BF16_DMA, kBf16Tile, kBf16Tile, kBf16DmaK}
                : GemmTile{GV_BF16_REG, kBf16Tile, kBf16Tile, kBf16RegK};
}

}  // namespace jh
