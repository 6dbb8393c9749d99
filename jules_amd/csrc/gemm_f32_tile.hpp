// gemm_f32_tile.hpp - fp32 GEMM tiles on the fp32 MFMAs.
//
// C [M,N] = epilogue(op(A) [M,K] . op(B) [K,N]), op(X) = X^T with TA / TB.
//
// v_mfma_f32_32x32x2_f32 and v_mfma_f32_16x16x4_f32 compute each output as a
// chain of correctly rounded fmas over k in ascending order: their results are
// the bits of acc = fmaf(a[k], b[k], acc) for k = 0, 1, .. on random operands,
// operands whose products or sums are subnormal, overflow, or hold infinities,
// NaNs and signed zeros (500 000 outputs compared, none different).  So a tile
// that walks k in order without splitting it gives the reference's fma chain
// bit for bit, at the matrix cores' rate: 157 TFLOP/s, twice what v_fma_f32
// reaches.  k past K takes a = +0, b = -0: fmaf(+0, -0, acc) is acc for every
// acc, -0 included.
//
// A workgroup of 2 x 2 waves owns a BM x BN tile, a wave MT x NT accumulators
// of MF x MF.  Slices of BK k go global -> registers -> LDS, double-buffered,
// the loads of the next PF slices in flight during the current one's MFMAs, one
// barrier per slice.  The MFMAs are slow against their operands' traffic (64 cycles
// for two 4-byte values a lane), so LDS and loads are not what binds; what
// does is how evenly the tiles fill 256 CUs, and for small problems the chain
// itself: K MFMA latencies (16 x 16: 8 cycles a k; 32 x 32: 32).
//
// An MFMA wants k = KP j + p from lane group p = lane / MF.  An operand whose
// k is contiguous in memory is kept as rows of k, the KP residues apart, so
// one 16-byte read feeds four MFMAs; an operand whose k is the outer dimension
// is kept as it is, rows padded so that the lane groups' rows (KP of them) lie
// in different banks.
#pragma once

#include <type_traits>

#include "common.hpp"
#include "launch.hpp"

namespace jh {

// acc += A . B over one MFMA of MF x MF
template <int MF>
struct F32Mfma;
template <>
struct F32Mfma<32> {
    typedef float Acc __attribute__((ext_vector_type(16)));
    static constexpr int KP = 2, NR = 16;
    static __device__ __forceinline__ Acc run(float a, float b, Acc c) {
        return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int lane, int e) { return 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3); }
};
template <>
struct F32Mfma<16> {
    typedef float Acc __attribute__((ext_vector_type(4)));
    static constexpr int KP = 4, NR = 4;
    static __device__ __forceinline__ Acc run(float a, float b, Acc c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int lane, int e) { return 4 * (lane >> 4) + e; }
};

// One operand's slice, X rows (columns) of the tile by BK k.  CONTIG: k is the
// contiguous dimension in memory, loaded 4 floats at a time wherever the rows
// start (only the last slice, one float at a time, can reach past a row).  Else
// V = 4 needs the number of rows to be a multiple of 4, so that a piece is
// wholly inside or outside, and V = 1 does not; V = 0 is 1 with 64-bit offsets.
template <int MF, int X, int BK, bool CONTIG, int V_, bool IS_B>
struct F32Slice {
    static constexpr bool BIG = V_ == 0;
    static constexpr int V = CONTIG ? 4 : BIG ? 1 : V_;
    static constexpr int KP = F32Mfma<MF>::KP;
    static constexpr int PITCH = CONTIG ? BK + 4 : X + MF;
    static constexpr int FLOATS = CONTIG ? X * PITCH : BK * PITCH;
    static constexpr int NP = X * BK / V / 256;  // loads per thread
    static_assert(NP * V * 256 == X * BK, "whole loads per thread");
    float r[NP * V];

    static __device__ __forceinline__ int x_of(int p) {
        const int i = threadIdx.x + 256 * p;
        return CONTIG ? i / (BK / V) : i % (X / V) * V;
    }
    static __device__ __forceinline__ int k_of(int p) {
        const int i = threadIdx.x + 256 * p;
        return CONTIG ? i % (BK / V) * V : i / (X / V);
    }
    // Where a thread's loads of a whole slice start: a base for the workgroup,
    // advanced by the slice on the scalar unit, and a 32-bit byte offset per
    // load (64-bit pointers took as many VALU cycles per slice as a 32 x 32
    // tile's MFMAs).  BIG: the tile spans 2^32 bytes or more, 64-bit offsets.
    // Rows past xn repeat the last: their outputs are not stored.
    using Off = std::conditional_t<BIG, int64_t, uint32_t>;
    struct Src {
        const char* base;
        Off o[NP];
        __device__ __forceinline__ Src(const float* P, int64_t ld, int x0, int xn, int k0) {
            const int last = xn - (CONTIG ? 1 : V), xb = min(x0, last);
            base = reinterpret_cast<const char*>(CONTIG ? P + xb * ld + k0 : P + k0 * ld + xb);
#pragma unroll
            for (int p = 0; p < NP; ++p) {
                const Off x = (Off)(min(x0 + x_of(p), last) - xb), k = (Off)k_of(p);
                o[p] = (CONTIG ? x * (Off)ld + k : k * (Off)ld + x) * 4;
            }
        }
        __device__ __forceinline__ const float* at(int p) const {
            return reinterpret_cast<const float*>(base + o[p]);
        }
    };
    static __device__ __forceinline__ f32x4_t get4(const float* q) {
        return reinterpret_cast<const f32x4_any_t*>(q)->v;
    }
    // the next slice, k0 .. k0 + BK, of which the k below kn exist
    __device__ __forceinline__ void load(Src& s, int64_t ld, int k0, int kn) {
        if (k0 + BK <= kn) {
#pragma unroll
            for (int p = 0; p < NP; ++p) {
                if constexpr (V == 4) {
                    const f32x4_t v = get4(s.at(p));
#pragma unroll
                    for (int e = 0; e < 4; ++e) r[4 * p + e] = v[e];
                } else {
                    r[p] = *s.at(p);
                }
            }
            s.base += 4 * (CONTIG ? (int64_t)BK : BK * ld);
            return;
        }
        // the last slice: k past kn are read from the last k instead, and
        // replaced
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            const int k = k0 + k_of(p);
            if constexpr (CONTIG) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float v = *(s.at(p) + (min(k + e, kn - 1) - k));
                    r[4 * p + e] = k + e < kn ? v : (IS_B ? -0.0f : 0.0f);
                }
            } else {
                const float* q = s.at(p) + (min(k, kn - 1) - k) * ld;
                if constexpr (V == 4) {
                    const f32x4_t v = get4(q);
#pragma unroll
                    for (int e = 0; e < 4; ++e) r[4 * p + e] = v[e];
                } else {
                    r[p] = *q;
                }
#pragma unroll
                for (int e = 0; e < V; ++e) r[V * p + e] = k < kn ? r[V * p + e] : (IS_B ? -0.0f : 0.0f);
            }
        }
    }
    // row x of the slice = 1
    __device__ __forceinline__ void fill_row(int x) {
#pragma unroll
        for (int p = 0; p < NP; ++p)
#pragma unroll
            for (int e = 0; e < V; ++e) r[V * p + e] = x_of(p) + (CONTIG ? 0 : e) == x ? 1.0f : r[V * p + e];
    }
    __device__ __forceinline__ void store(float* s) const {
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            const int x = x_of(p), k = k_of(p);
            if constexpr (!CONTIG) {
                float* d = s + k * PITCH + x;
                if constexpr (V == 4) *reinterpret_cast<f32x4_t*>(d) = f32x4_t{r[4 * p], r[4 * p + 1], r[4 * p + 2], r[4 * p + 3]};
                else *d = r[p];
            } else if constexpr (V == 4 && KP == 2) {
                float* d = s + x * PITCH + k / 2;
                *reinterpret_cast<f32x2_t*>(d) = f32x2_t{r[4 * p], r[4 * p + 2]};
                *reinterpret_cast<f32x2_t*>(d + BK / 2) = f32x2_t{r[4 * p + 1], r[4 * p + 3]};
            } else {
#pragma unroll
                for (int e = 0; e < V; ++e) s[x * PITCH + (k + e) % KP * (BK / KP) + (k + e) / KP] = r[V * p + e];
            }
        }
    }
    // the operand of MFMAs 4 g .. 4 g + 3 for this lane: row x of the slice
    static __device__ __forceinline__ f32x4_t frag(const float* s, int x, int ph, int g) {
        if constexpr (CONTIG) {
            return *reinterpret_cast<const f32x4_t*>(s + x * PITCH + ph * (BK / KP) + 4 * g);
        } else {
            const float* d = s + (4 * KP * g + ph) * PITCH + x;
            return f32x4_t{d[0], d[KP * PITCH], d[2 * KP * PITCH], d[3 * KP * PITCH]};
        }
    }
};

// A barrier that orders LDS only: __syncthreads() would also wait for the
// slices still being loaded.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <int MF, int MT, int NT, int BK, int PF, bool TA, bool TB, int V, bool FOLD = false>
struct F32Tile {
    using Mf = F32Mfma<MF>;
    static constexpr int BM = 2 * MT * MF, BN = 2 * NT * MF, KP = Mf::KP;
    using SA = F32Slice<MF, BM, BK, !TA, V, false>;
    using SB = F32Slice<MF, BN, BK, TB, V, true>;
    static constexpr int STAGE = SA::FLOATS + SB::FLOATS;

    // acc = the tile at (m0, n0) over k in [kb, ke).  FOLD (chunk > 0, a
    // multiple of 16; one accumulator a wave only; a kernel of its own, its test
    // per four k-steps costs a chain 12 %): the sum is taken over chunks of that
    // many k, each its own chain, added in order, as a K split into ranges of
    // chunk would add its partial sums.  ones: row M of op(A) reads as 1, so
    // output row M is the column sum of op(B) (TA only).
    static __device__ __forceinline__ void run(const float* A, int64_t lda, const float* B, int64_t ldb, int m0,
                                               int M, int n0, int N, int kb, int ke, int chunk, bool ones,
                                               float* sm, typename Mf::Acc (&acc)[MT][NT]) {
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        const int xa = (wave >> 1) * MT * MF + lane % MF, xb = (wave & 1) * NT * MF + lane % MF, ph = lane / MF;
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) acc[i][j] = typename Mf::Acc{};
        if (kb >= ke) return;
        // While slice t is multiplied, slice t + 1 goes from its registers to
        // the other LDS buffer (free since the last barrier).  One accumulator:
        // first of all, then slice t + 1 + PF is loaded into them, and the
        // operands of four k-steps are read during the MFMAs of the four before.
        // With more the compiler's own order is the better one (4096^3 at 128 x
        // 128 1046 against 1374 us): slice t + PF loaded first, slice t + 1
        // stored last.
        constexpr bool AHEAD = MT * NT == 1;
        static_assert(AHEAD || !FOLD, "one accumulator");
        SA ra[PF];
        SB rb[PF];
        typename SA::Src pa(A, lda, m0, M, kb);
        typename SB::Src pb(B, ldb, n0, N, kb);
        auto load = [&](int u, int k0) {
            if (k0 >= ke) return;
            ra[u].load(pa, lda, k0, ke);
            rb[u].load(pb, ldb, k0, ke);
            if constexpr (TA)
                if (ones) ra[u].fill_row(M - m0);
        };
        auto store = [&](int u, int b) {
            ra[u].store(sm + b * STAGE);
            rb[u].store(sm + b * STAGE + SA::FLOATS);
        };
#pragma unroll
        for (int u = 0; u < PF; ++u) load(u, kb + u * BK);
        store(0, 0);
        if constexpr (AHEAD) load(0, kb + PF * BK);
        lds_barrier();
        int buf = 0, left = chunk;
        bool first = true;
        typename Mf::Acc tot[MT][NT];
        auto fold = [&]() {
            tot[0][0] = first ? acc[0][0] : tot[0][0] + acc[0][0];
            acc[0][0] = typename Mf::Acc{};
            first = false;
            left = chunk;
        };
        for (int kt = kb; kt < ke; kt += PF * BK) {
#pragma unroll
            for (int u = 0; u < PF; ++u) {
                const int k0 = kt + u * BK;
                if (k0 >= ke) break;
                const float* sa = sm + buf * STAGE;
                const float* sb = sa + SA::FLOATS;
                buf ^= 1;
                constexpr int NG = BK / KP / 4;
                f32x4_t a[2][MT], b[2][NT];
                auto read = [&](int g) {
#pragma unroll
                    for (int i = 0; i < MT; ++i) a[g & 1][i] = SA::frag(sa, xa + i * MF, ph, g);
#pragma unroll
                    for (int j = 0; j < NT; ++j) b[g & 1][j] = SB::frag(sb, xb + j * MF, ph, g);
                };
                if constexpr (AHEAD) read(0);
                else load(u, k0 + PF * BK);
#pragma unroll
                for (int g = 0; g < NG; ++g) {
                    if constexpr (!AHEAD) read(g);
                    else if (g + 1 < NG) read(g + 1);
                    if constexpr (AHEAD) {
                        if (g == 0) {
                            if (k0 + BK < ke) store((u + 1) % PF, buf);
                            load((u + 1) % PF, k0 + (PF + 1) * BK);
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
#pragma unroll
                    for (int s = 0; s < 4; ++s)
#pragma unroll
                        for (int i = 0; i < MT; ++i)
#pragma unroll
                            for (int j = 0; j < NT; ++j)
                                acc[i][j] = Mf::run(a[g & 1][i][s], b[g & 1][j][s], acc[i][j]);
                    if constexpr (AHEAD) {
                        __builtin_amdgcn_sched_barrier(0);
                        if constexpr (FOLD)
                            if (k0 + 4 * KP * g < ke && (left -= 4 * KP) == 0) fold();
                    }
                }
                if (!AHEAD && k0 + BK < ke) store((u + 1) % PF, buf);
                lds_barrier();
            }
        }
        if constexpr (FOLD) {
            if (left != chunk) fold();
            acc[0][0] = tot[0][0];
        }
    }
};

}  // namespace jh
