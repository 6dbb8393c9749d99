// gemm_tile.hpp - the main loop of the MFMA GEMMs at any shape whose rows are
// whole 16-byte pieces: bf16 (gemm_bf16.hip) and int8 (matmul_int8.hip).
//
// C tile [BM x BN] = A [M,K] . B [K,N], both row-major, WM x WN x KG waves, each
// wave MT x NT accumulators of 32 x 32 over every KG-th k-step.  One k-step is 32 bytes of an A row
// (16 bf16 or 32 int8) and feeds one MFMA per accumulator; a slice is RB bytes
// of every A row (KS = RB / 32 k-steps) and the same number of B rows.
//
// Slices reach LDS by LDS DMA through a ring of NST stages.  The copies are
// range-checked buffer loads, so ragged shapes need no second kernel: a row
// past M, a B row past K or a 16-byte piece past the end of A's rows reads 0
// (K past its end must be 0 on both sides, or an infinity in the next row of
// A would meet the 0 of B); a column past N reads whatever follows and only
// feeds outputs that are not stored.  The resources move with the slice, so
// the lanes' offsets are computed once.  Slices past the last have an empty
// range: every trip of the loop issues the same copies, and every wait count
// is a constant.
//
//   A stage: rows of RB bytes, 16-byte piece c of row r at
//      c ^ ((r >> 1) & 7) (RB = 128) or c ^ ((r >> 2) & 3) (RB = 64): a
//      fragment read (ds_read_b128, 16 consecutive rows, one piece) touches
//      16 distinct 16-byte groups of the 64 banks.
//   B stage: rows of BN elements, 32-byte block b of row r at b ^ f(r)
//      (b_swz): the rows that one transposing read serves together (4 rows x
//      64 bytes for ds_read_b64_tr_b16, 8 rows x 32 bytes for
//      ds_read_b64_tr_b8) cover all 64 banks.
//
// LDS reads are inline asm with explicit lgkmcnt waits (through the builtins
// the compiler drains every copy in flight before a transposing read).  They
// run PF k-steps ahead of the MFMAs that use them, in a ring of fragment
// registers of its own (SLOTS > PF, so no read lands in a slot whose MFMAs
// are still to issue).
#pragma once

#include <type_traits>
#include <utility>

#include "common.hpp"
#include "launch.hpp"

namespace jh {

typedef int i32x16_t __attribute__((ext_vector_type(16)));
typedef int i32x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_ptr_t;

template <int I, int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N>(f);
    }
}

struct Bf16Op {
    static constexpr int ES = 2;       // bytes per element
    static constexpr int TR_ROWS = 4;  // k rows one transposing read covers
    using Acc = f32x16_t;
    static __device__ __forceinline__ u32x2_t read_tr(uint32_t a) {
        u32x2_t v;
        asm volatile("ds_read_b64_tr_b16 %0, %1" : "=v"(v) : "v"(a) : "memory");
        return v;
    }
    static __device__ __forceinline__ Acc mfma(u32x4_t a, u32x4_t b, Acc c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                       __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
    }
};

struct Int8Op {
    static constexpr int ES = 1;
    static constexpr int TR_ROWS = 8;
    using Acc = i32x16_t;
    static __device__ __forceinline__ u32x2_t read_tr(uint32_t a) {
        u32x2_t v;
        asm volatile("ds_read_b64_tr_b8 %0, %1" : "=v"(v) : "v"(a) : "memory");
        return v;
    }
    static __device__ __forceinline__ Acc mfma(u32x4_t a, u32x4_t b, Acc c) {
        return __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(i32x4_t, a),
                                                     __builtin_bit_cast(i32x4_t, b), c, 0, 0, 0);
    }
};

__device__ __forceinline__ u32x4_t tile_read_b128(uint32_t a) {
    u32x4_t v;
    asm volatile("ds_read_b128 %0, %1" : "=v"(v) : "v"(a) : "memory");
    return v;
}

// The fragments of one k-step, and the wait that orders their use: at most N
// LDS reads outstanding, the registers passing through the asm so that no
// MFMA that uses them is scheduled before it.
template <int MT, int NT>
struct TileFrags {
    u32x4_t a[MT];
    u32x2_t b[NT][2];  // the two transposing reads of each B fragment
    template <int N>
    __device__ __forceinline__ void wait() {
        static_assert(N >= 0 && N <= 15, "lgkmcnt is a 4-bit count");
        asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(N) : "memory");
#pragma unroll
        for (int i = 0; i < MT; ++i) asm volatile("" : "+v"(a[i])::"memory");
#pragma unroll
        for (int j = 0; j < NT; ++j) asm volatile("" : "+v"(b[j][0]), "+v"(b[j][1])::"memory");
    }
    __device__ __forceinline__ u32x4_t bfrag(int j) const {
        return u32x4_t{b[j][0][0], b[j][0][1], b[j][1][0], b[j][1][1]};
    }
};

template <class OP_, int BM_, int BN_, int WM_, int WN_, int KG_, int RB_, int NST_, int PF_>
struct TileCfg {
    using OP = OP_;
    static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_, KG = KG_, RB = RB_, NST = NST_, PF = PF_;
    static constexpr int NW = WM * WN * KG, THREADS = 64 * NW;
    static constexpr int MT = BM / WM / 32, NT = BN / WN / 32;
    static constexpr int ES = OP::ES;
    static constexpr int BK = RB / ES;              // k per slice
    static constexpr int KS = RB / 32 / KG;         // k-steps per slice and wave
    static constexpr int BRB = BN * ES;             // bytes of a B row in LDS
    static constexpr int A_BYTES = BM * RB, B_BYTES = BK * BRB, STAGE = A_BYTES + B_BYTES;
    static constexpr int LDS = NST * STAGE;
    static constexpr int PA = A_BYTES / 1024 / NW, PB = B_BYTES / 1024 / NW, PPS = PA + PB;
    static constexpr int RPS = MT + 2 * NT;         // LDS reads of a k-step
    static constexpr int SLOTS = KS;
    static constexpr int OWN = MT * NT / KG;        // accumulators a wave finishes
    static_assert(OWN * KG == MT * NT, "whole accumulators per wave");
    static_assert(KG == 1 || WM * WN * KG * (MT * NT - OWN) * 4096 <= NST * STAGE, "exchange space");
    static_assert(PA * NW * 1024 == A_BYTES && PB * NW * 1024 == B_BYTES, "whole copies per wave");
    static_assert(PF >= 1 && PF < KS && RPS * (PF - 1) <= 15 && NST >= 3, "look-ahead");
    static_assert((NST - 2) * PPS <= 63, "vmcnt is a 6-bit count");
    static_assert(LDS <= 160 * 1024, "LDS of a CU");
    using Acc = typename OP::Acc;

    static __device__ __forceinline__ int a_swz(int r) { return RB == 128 ? (r >> 1) & 7 : (r >> 2) & 3; }
    // what 32-byte block b of B row r is XORed with
    static __device__ __forceinline__ int b_swz(int r) {
        if constexpr (OP::TR_ROWS == 4) return BRB >= 256 ? 2 * (r & 3) : 2 * ((r >> 1) & 1);
        else return BRB >= 256 ? (r & 7) : BRB == 128 ? (r >> 1) & 3 : (r >> 2) & 1;
    }

    // own = the k range [0, kn) of this tile, summed.  A: row m0 at the range's first
    // k, lda bytes between rows, `rows` of them valid; B: column n0 of the
    // range's first row, ldb bytes between rows, `colb` bytes valid to the end
    // of a row.  sm: LDS bytes, 1 KiB aligned.  rows * lda and BK * ldb stay
    // below 2^31 (the caller's rule).
    static __device__ __forceinline__ void run(const uint8_t* A, int64_t lda, int rows, const uint8_t* B,
                                               int64_t ldb, int64_t colb, int kn, uint8_t* sm,
                                               Acc (&own)[OWN]) {
        Acc acc[MT][NT];
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) acc[i][j] = Acc{};
        const int lane = threadIdx.x & 63;
        const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
        constexpr uint32_t OOB = 0x80000000u;
        constexpr int APR = RB / 16, BPR = BRB / 16;  // 16-byte pieces per row

        // lane offsets of this wave's copies (segment i * NW + wave, 1 KiB)
        uint32_t a_off[PA], b_off[PB];
        int a_k[PA];  // byte of the A row within the slice
#pragma unroll
        for (int i = 0; i < PA; ++i) {
            const int u = (i * NW + wave) * 64 + lane, r = u / APR;
            a_k[i] = ((u % APR) ^ a_swz(r)) * 16;
            a_off[i] = r < rows ? (uint32_t)r * (uint32_t)lda + a_k[i] : OOB;
        }
#pragma unroll
        for (int i = 0; i < PB; ++i) {
            const int u = (i * NW + wave) * 64 + lane, r = u / BPR, c = u % BPR;
            const int lc = ((((c >> 1) ^ b_swz(r)) << 1) | (c & 1)) * 16;
            b_off[i] = (uint32_t)r * (uint32_t)ldb + lc;
        }
        const uint32_t a_range = (uint32_t)rows * (uint32_t)lda;
        auto copy = [&](int kt, int p) {
            uint8_t* st = sm + (kt % NST) * STAGE;
            const int k0 = kt * BK;
            if (p < PA) {
                const int kleft = (kn - k0) * ES;  // bytes of the A rows left
                const __amdgpu_buffer_rsrc_t src = __builtin_amdgcn_make_buffer_rsrc(
                    const_cast<uint8_t*>(A) + (int64_t)k0 * ES, 0, a_range, 0x00020000);
                const uint32_t o = a_k[p] < kleft ? a_off[p] : OOB;
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    src, (lds_ptr_t*)(st + (p * NW + wave) * 1024), 16, o, 0, 0, 0);
            } else {
                const int left = min(BK, kn - k0);
                const int64_t bytes = (int64_t)(left - 1) * ldb + min((int64_t)colb, ldb);
                const __amdgpu_buffer_rsrc_t src = __builtin_amdgcn_make_buffer_rsrc(
                    const_cast<uint8_t*>(B) + (int64_t)k0 * ldb, 0, left > 0 ? (uint32_t)bytes : 0u,
                    0x00020000);
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    src, (lds_ptr_t*)(st + A_BYTES + ((p - PA) * NW + wave) * 1024), 16,
                    b_off[p - PA], 0, 0, 0);
            }
        };

        // LDS addresses of the reads of k-step 0; a k-step adds 2 pieces to A
        // (before its swizzle) and 2 or 4 * TR_ROWS rows to B
        const int wm = wave / WN % WM, wn = wave % WN, kg = wave / (WM * WN);
        const int fr = lane & 31, half = lane >> 5, ts = lane & 15, tdh = (lane >> 4) & 1;
        const uint32_t s0 = (uint32_t)(uintptr_t)sm;
        uint32_t ra[KS][MT], rb[NT][2];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                const int r = (wm * MT + i) * 32 + fr;
                ra[ks][i] = s0 + r * RB + (((2 * (ks * KG + kg) + half) ^ a_swz(r)) << 4);
            }
        // B: lane s of a 16-lane group addresses row s / LPR, 8-byte piece s % LPR
        // of the group's 16 columns
        constexpr int LPR = 16 / OP::TR_ROWS;
        constexpr int KROWS = 32 / ES;  // k rows of a k-step
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int r = (KROWS / 2) * half + OP::TR_ROWS * h + ts / LPR;
                const int cb = ((wn * NT + j) * 32 + 16 * tdh) * ES + (ts % LPR) * 8;
                rb[j][h] = s0 + A_BYTES + kg * KROWS * BRB + r * BRB + (((cb >> 5) ^ b_swz(r)) << 5) + (cb & 31);
            }
        TileFrags<MT, NT> f[SLOTS];
        // read q of k-step ks (compile time) of the slice at stage offset so
        auto read = [&](auto ksc, int q, uint32_t so) {
            constexpr int ks = decltype(ksc)::value;
            if (q < MT) {
                f[ks].a[q] = tile_read_b128(ra[ks][q] + so);
            } else {
                // b_swz repeats every KROWS rows, so a k-step only adds to the address
                const int j = (q - MT) >> 1, h = (q - MT) & 1;
                f[ks].b[j][h] = OP::read_tr(rb[j][h] + so + ks * KG * KROWS * BRB);
            }
        };

        const int KT = (kn + BK - 1) / BK;
#pragma unroll
        for (int p = 0; p < NST - 1; ++p)
#pragma unroll
            for (int q = 0; q < PPS; ++q) copy(p, q);
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NST - 2) * PPS) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        static_for<0, PF>([&](auto ks) {
#pragma unroll
            for (int q = 0; q < RPS; ++q) read(ks, q, 0);
        });

        constexpr int MM = MT * NT;       // MFMAs of a k-step
        constexpr int DMA_SLOTS = PF * MM;  // MFMAs that a slice's copies are spread over
        uint32_t cur = 0;                 // stage offset of slice kt
        for (int kt = 0; kt < KT; ++kt) {
            const uint32_t nxt = cur + STAGE == (uint32_t)LDS ? 0u : cur + STAGE;
            static_for<0, KS>([&](auto sc) {
                constexpr int s = decltype(sc)::value;
                constexpr int ahead = (s + PF) % KS;  // k-step read during this one
                if constexpr (s == KS - PF) {
                    // Slice kt + 1 has landed once only the copies of the slices
                    // after it remain (slices up to kt + NST - 2 are issued).
                    // The barrier also ends every wave's reads of slice kt - 1,
                    // whose stage the copies below refill.
                    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NST - 3) * PPS) : "memory");
                    __builtin_amdgcn_s_barrier();
                    asm volatile("" ::: "memory");
                }
                f[s].template wait<RPS*(PF - 1)>();
                const uint32_t so = s + PF >= KS ? nxt : cur;
#pragma unroll
                for (int i = 0; i < MM; ++i) {
                    acc[i / NT][i % NT] =
                        OP::mfma(f[s].a[i / NT], f[s].bfrag(i % NT), acc[i / NT][i % NT]);
#pragma unroll
                    for (int q = i * RPS / MM; q < (i + 1) * RPS / MM; ++q)
                        read(std::integral_constant<int, ahead>{}, q, so);
                    if constexpr (s >= KS - PF) {
                        const int d = (s - (KS - PF)) * MM + i;
#pragma unroll
                        for (int q = d * PPS / DMA_SLOTS; q < (d + 1) * PPS / DMA_SLOTS; ++q)
                            copy(kt + NST - 1, q);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            });
            cur = nxt;
        }
        // the reads ahead of the last k-step and the copies past the last slice
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        static_for<0, SLOTS>([&](auto sc) { f[decltype(sc)::value].template wait<0>(); });

        // Sum over the k groups: a wave keeps accumulators [kg * OWN, kg * OWN +
        // OWN) and hands the others to the waves that keep them, through LDS,
        // added in group order.
        if constexpr (KG == 1) {
#pragma unroll
            for (int t = 0; t < OWN; ++t) own[t] = acc[t / NT][t % NT];
        } else {
            __syncthreads();
            typedef decltype(acc[0][0][0] + acc[0][0][0]) E;
            typedef E E4 __attribute__((ext_vector_type(4)));
            const int wmn = wave % (WM * WN);
            // part of group `from` for the t-th accumulator kept by group `to`
            auto slot = [&](int from, int to, int t) {
                const int c = from < to ? from : from - 1;
                return reinterpret_cast<E4*>(sm) + ((((wmn * KG + to) * (KG - 1) + c) * OWN + t) * 4) * 64 + lane;
            };
            static_for<0, KG>([&](auto gc) {
                constexpr int to = decltype(gc)::value;
                if (kg == to) return;
#pragma unroll
                for (int t = 0; t < OWN; ++t)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const Acc& v = acc[(to * OWN + t) / NT][(to * OWN + t) % NT];
                        slot(kg, to, t)[64 * q] = E4{v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
                    }
            });
            __syncthreads();
            static_for<0, KG>([&](auto gc) {
                constexpr int g = decltype(gc)::value;
                if (kg != g) return;
#pragma unroll
                for (int t = 0; t < OWN; ++t) {
                    const Acc& mine = acc[(g * OWN + t) / NT][(g * OWN + t) % NT];
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        E4 v = E4{mine[4 * q], mine[4 * q + 1], mine[4 * q + 2], mine[4 * q + 3]};
                        if constexpr (g > 0) {
                            E4 sum = slot(0, g, t)[64 * q];
#pragma unroll
                            for (int o = 1; o < g; ++o) sum += slot(o, g, t)[64 * q];
                            v = sum + v;
                        }
#pragma unroll
                        for (int o = g + 1; o < KG; ++o) v += slot(o, g, t)[64 * q];
#pragma unroll
                        for (int x = 0; x < 4; ++x) own[t][4 * q + x] = v[x];
                    }
                }
            });
        }
    }

    // row and column within the tile of element e of own[t]
    static __device__ __forceinline__ int own_row(int t, int e) {
        const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
        const int i = (wave / (WM * WN) * OWN + t) / NT;
        return (wave / WN % WM * MT + i) * 32 + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3);
    }
    static __device__ __forceinline__ int own_col(int t) {
        const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
        const int j = (wave / (WM * WN) * OWN + t) % NT;
        return (wave % WN * NT + j) * 32 + (lane & 31);
    }
};

// Output tile and split of a workgroup.  Workgroup ids go to the 8 XCDs round
// robin; each XCD gets a contiguous run of (split, tile), tiles in bands of GM
// rows of tiles walked column by column, so that the workgroups an XCD runs
// at once share A rows and B columns in its L2.
struct TileCoord {
    int tm, tn, z;
};
template <int GM>
__device__ __forceinline__ TileCoord tile_coord(int tiles_m, int tiles_n) {
    const int nblk = gridDim.x, per = nblk >> 3, rest = nblk & 7;
    const int x = blockIdx.x & 7, i = blockIdx.x >> 3;
    int t = x * per + min(x, rest) + i;
    const int tiles = tiles_m * tiles_n;
    const int z = t / tiles;
    t -= z * tiles;
    const int band = t / (GM * tiles_n), first = band * GM;
    const int gs = min(GM, tiles_m - first), in = t - band * GM * tiles_n;
    return {first + in % gs, in / gs, z};
}

// Which tile and how many K ranges a launch takes: the least of a cost model
// over the tiles.  `wg` workgroups over kc elements each take about
//   base + rounds * (kc * per_k * (1 + fill * min(1, wg / 256)) + round) us,
// rounds = ceil(wg / 256), times `shared` where two workgroups share a CU, and
// S K ranges add split_base + split_z S + split_mn S M N us for the partial
// sums and their reduction.  Each operand type has its own constants, fitted
// to measured times (gemm_bf16.hip, matmul_int8.hip).
struct TilePlan {
    int bm, bn, bk, threads;
    float base, per_k, round, shared;
};
struct TileModel {
    TilePlan plan[6];
    float fill, split_base, split_z, split_mn;
};
struct TileChoice {
    int plan, splits, kc;
};

inline TileChoice tile_choice(const TileModel& m, int M, int N, int K, bool may_split) {
    TileChoice best{0, 1, 0};
    float best_us = 0.0f;
    for (int c = 0; c < 6; ++c) {
        const TilePlan& p = m.plan[c];
        const int64_t tiles = (((int64_t)M + p.bm - 1) / p.bm) * (((int64_t)N + p.bn - 1) / p.bn);
        // the runtime takes fewer than 2^32 threads a launch (split ones are few)
        if (tiles * p.threads >= int64_t(1) << 32 && c < 5) continue;
        const int slices = (K + p.bk - 1) / p.bk;
        for (int S : {1, 2, 3, 4, 6, 8}) {
            if (S > 1 && (!may_split || slices < 2 * S || tiles * S > 512 ||
                          (int64_t)S * M * N * 4 > (int64_t)kMaxPartialBytes))
                break;
            const int per = (slices + S - 1) / S;
            const int z = slices ? (slices + per - 1) / per : 1;
            const int64_t wg = tiles * z;
            const float rounds = (float)((wg + 255) / 256);
            const float per_k = p.per_k * (1.0f + m.fill * (wg < 256 ? (float)wg / 256.0f : 1.0f));
            float us = p.base + (rounds > 1.0f ? rounds * p.shared : 1.0f) *
                                    ((float)per * (float)p.bk * per_k + p.round);
            if (z > 1) us += m.split_base + m.split_z * z + m.split_mn * z * M * N;
            if (best_us == 0.0f || us < best_us) {
                best_us = us;
                best = {c, z, per * p.bk};
            }
        }
    }
    return best;
}

// tile_choice with the partial sums' memory: the stream's buffer for them,
// under its lock until the caller has enqueued the reduction.  It may not be
// allocated while a graph is being captured, nor kept by the graph (eager calls
// on the stream write it while the graph may run on another), and
// hipStreamPerThread is one handle for many streams: there, and without memory
// for it, K is not split.
inline TileChoice tile_plan(const TileModel& m, int M, int N, int K, hipStream_t s, void** part,
                            WorkspaceLock* lock) {
    *part = nullptr;
    TileChoice c = tile_choice(m, M, N, K, s != hipStreamPerThread);
    if (c.splits == 1) return c;
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &cap) == hipSuccess && cap == hipStreamCaptureStatusNone) {
        // another thread may be capturing: allocating the buffer concerns this
        // stream only, and must not end that capture
        hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
        (void)hipThreadExchangeStreamCaptureMode(&mode);
        const hipError_t e = stream_partials(s, part, lock);
        (void)hipThreadExchangeStreamCaptureMode(&mode);
        if (e == hipSuccess) return c;
    }
    (void)hipGetLastError();
    *part = nullptr;
    return tile_choice(m, M, N, K, false);
}

}  // namespace jh
