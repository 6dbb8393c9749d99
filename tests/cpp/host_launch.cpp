// host_launch.cpp - what the library's entry points launch, and what they do
// with the workspaces they hold, checked without a GPU: the library's host code,
// launchers included, built with AddressSanitizer and UndefinedBehaviorSanitizer
// and linked against hip_stub.cpp.  `host_launch <check>` runs one check and prints
// "<check> ok"; run by tests/test_host_launch.py.
#include <algorithm>
#include <chrono>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <future>
#include <iostream>
#include <sstream>
#include <string>
#include <vector>

#include "hip_stub.hpp"
#include "jules_hip.h"
#include "jules_hip_kernel.hpp"
#include "launch.hpp"

static int g_fail = 0;
#define EXPECT(cond, ...)                                                            \
    do {                                                                             \
        if (!(cond)) {                                                               \
            if (++g_fail <= 20) {                                                    \
                std::fprintf(stderr, "line %d: expected %s: ", __LINE__, #cond);     \
                std::fprintf(stderr, __VA_ARGS__);                                   \
                std::fprintf(stderr, "\n");                                          \
            }                                                                        \
        }                                                                            \
    } while (0)

// an operand that no check lets anything read
template <typename T = float>
static T* fake(int i) {
    return reinterpret_cast<T*>((uintptr_t(1) << 46) + (uintptr_t(i) << 42));
}

// A launch of the fp32 tile kernel: its tile and variant, from its name.
struct F32Launch {
    int mf, mt, nt, bk, pf, v;
    bool ta, tb, fold;
};
static bool f32_launch(const std::string& name, F32Launch* f) {
    char ta[8], tb[8], fold[8];
    const int n = std::sscanf(name.c_str(),
                              "void jh::gemm_f32_tile_kernel<jh::F32Cfg<%d, %d, %d, %d, %d>, %5[a-z], %5[a-z], %d, %5[a-z]>",
                              &f->mf, &f->mt, &f->nt, &f->bk, &f->pf, ta, tb, &f->v, fold);
    f->ta = !std::strcmp(ta, "true");
    f->tb = !std::strcmp(tb, "true");
    f->fold = !std::strcmp(fold, "true");
    return n == 9;
}

// Every fp32 product whose tile spans 2^32 bytes of an operand takes the 64-bit
// offsets (V = 0).  The kernel forms an offset for each k of a slice, also those
// past K, of an operand whose k is the outer dimension, and for each row that
// exists of the others.
static void f32_offsets() {
    int tiles = 0, wide = 0;
    stub::on_launch = [&](const stub::Launch& l) {
        F32Launch f;
        if (!f32_launch(l.kernel, &f)) return;
        ++tiles;
        wide += f.v == 0;
        const auto g = l.arg<jh::F32Gemm>(0);
        const auto last = [&](bool k_outer, int x, int rows, int64_t ld) {
            const int64_t xs = std::min(x, rows);
            return 4 * (k_outer ? (f.bk - 1) * ld + xs : (xs - 1) * ld + f.bk);
        };
        const int64_t a = last(f.ta, 2 * f.mt * f.mf, g.M - (g.colsum ? 1 : 0), g.lda);
        const int64_t b = last(!f.tb, 2 * f.nt * f.mf, g.N, g.ldb);
        EXPECT(f.v == 0 || std::max(a, b) <= int64_t(1) << 32, "%s M=%d N=%d K=%d lda=%ld ldb=%ld", l.kernel.c_str(),
               g.M, g.N, g.K, (long)g.lda, (long)g.ldb);
        // and an ordinary row keeps the 32-bit ones
        EXPECT(f.v != 0 || std::max(g.lda, g.ldb) > 1 << 20, "%s lda=%ld ldb=%ld", l.kernel.c_str(), (long)g.lda,
               (long)g.ldb);
    };
    const int lds[] = {4096,     1 << 20,  8300000,  8388607,  8388608,   8400000,  8454659,  8454661, 9000000, 10000000,
                       16777215, 16777216, 16909321, 20000000, 33554432,  34636833, 67108863, 70000000, 71582789,
                       80000000, 300000000, 1 << 30, INT32_MAX};
    for (int ta : {0, 1})
        for (int tb : {0, 1})
            for (int M : {1, 3, 32, 33, 100, 512, 2048})
                for (int N : {1, 32, 33, 130, 2048})
                    for (int K : {1, 4, 10, 15, 17, 63, 64, 129, 256, 1024})
                        for (int ld : lds)
                            for (int other : {4096, ld}) {
                                const int lda = std::max(ld, ta ? M : K), ldb = std::max(other, tb ? K : N);
                                (void)jules_hip_sgemm(ta, tb, M, N, K, 1.0f, fake(0), lda, fake(1), ldb, 0.0f, fake(2),
                                                      N, nullptr);
                                const int la = std::max(other, ta ? M : K), lb = std::max(ld, tb ? K : N);
                                (void)jules_hip_sgemm(ta, tb, M, N, K, 1.0f, fake(0), la, fake(1), lb, 1.0f, fake(2),
                                                      N, nullptr);
                            }
    for (int M : {1, 8, 200})
        for (int K : {1, 4, 17, 40})
            for (int N : lds)
                (void)jules_hip_gemm_bias_act(JH_F32, JH_ACT_NONE, fake(0), fake(1), nullptr, fake(2), M, N, K, nullptr);
    for (int N : {1, 8, 200})
        for (int M : {1, 8, 200})
            for (int K : lds)
                (void)jules_hip_gemm_bias_act(JH_F32, JH_ACT_NONE, fake(0), fake(1), nullptr, fake(2), M, N, K, nullptr);
    EXPECT(tiles > 10000 && wide > 1000, "%d launches, %d with 64-bit offsets", tiles, wide);
}

// Calls that keep a workspace of the stream are run once, captured (their
// address is then the graph's) and followed by eager GEMMs that split K on the
// same stream: these may neither free nor use the memory that the graph holds.
static void graph_workspace() {
    const auto s = reinterpret_cast<hipStream_t>(uintptr_t(0x1230));
    const auto held = [&] {
        (void)jules_hip_flash_attn_fwd(JH_F32, 0, 0.1f, fake(0), fake(1), fake(2), fake(3), nullptr, 1, 2, 100, 80, s);
        (void)jules_hip_flash_attn_bwd(JH_BF16, 0, 0.1f, fake(0), fake(1), fake(2), fake(3), fake(4), fake(5), fake(6),
                                       fake(7), fake(8), 1, 2, 50, 80, fake(9), 1 << 20, s);
        (void)jules_hip_softmax(fake(0), fake(1), 2, 70000, s);
        (void)jules_hip_sgemm(0, 0, 64, 64, 4096, 1.0f, fake(0), 4096, fake(1), 64, 0.0f, fake(2), 64, s);
        (void)jules_hip_matmul_int8(fake<int8_t>(0), fake<int8_t>(1), fake(2), 8, 512, 1024, 1.0f, 1.0f, nullptr, s);
    };
    held();
    const auto before = stub::allocations();
    EXPECT(!before.empty(), "no workspace was allocated");
    stub::capturing.insert(s);
    int captured = 0;
    stub::on_launch = [&](const stub::Launch&) { ++captured; };
    held();
    EXPECT(captured > 10 && stub::allocations() == before, "%d launches captured", captured);
    stub::capturing.clear();

    int split = 0;
    stub::on_launch = [&](const stub::Launch& l) {
        const char* part = l.kernel.find("gemm_bf16_tile_kernel") != std::string::npos ? l.arg<const char*>(4)
                           : l.kernel.find("int8_tile_kernel") != std::string::npos    ? l.arg<const char*>(3)
                                                                                       : nullptr;
        if (!part) return;
        ++split;
        EXPECT(stub::allocated(part), "%s", l.kernel.c_str());
        for (const auto& b : before)
            EXPECT(part < b.first || part >= b.first + b.second, "%s writes the graph's workspace", l.kernel.c_str());
    };
    for (int N : {504, 1504, 4104}) {
        (void)jules_hip_gemm_bias_act(JH_BF16, JH_ACT_NONE, fake(0), fake(1), nullptr, fake(2), 24, N, 4352, s);
        (void)jules_hip_matmul_int8(fake<int8_t>(0), fake<int8_t>(1), fake(2), 72, N / 16 * 16, 4368, 1.0f, 1.0f,
                                    nullptr, s);
    }
    EXPECT(split >= 4, "%d GEMMs split K", split);
    for (const auto& b : before) EXPECT(stub::allocated(b.first), "the graph's workspace was freed");
}

// While a call waits for its stream to replace a workspace, calls of another
// thread on another stream go on.
static void stream_locks() {
    const auto a = reinterpret_cast<hipStream_t>(uintptr_t(0x1230)), b = reinterpret_cast<hipStream_t>(uintptr_t(0x4560));
    const auto decode = [](int N, hipStream_t s) {
        return jules_hip_matmul_int8(fake<int8_t>(0), fake<int8_t>(1), fake(2), 8, N, 1024, 1.0f, 1.0f, nullptr, s);
    };
    EXPECT(decode(512, a) == JH_OK, "first call");
    bool waited = false;
    stub::on_synchronize = [&](hipStream_t s) {
        if (s != a || waited) return;
        waited = true;
        auto other = std::async(std::launch::async, [&] {
            int st = decode(512, b);
            if (st == JH_OK) st = jules_hip_gemm_bias_act(JH_BF16, 0, fake(0), fake(1), nullptr, fake(2), 24, 504, 4352, b);
            return st;
        });
        if (other.wait_for(std::chrono::seconds(5)) != std::future_status::ready) {
            std::fprintf(stderr, "the other stream's calls wait too\n");
            std::_Exit(1);
        }
        EXPECT(other.get() == JH_OK, "calls on the other stream");
    };
    EXPECT(decode(8192, a) == JH_OK, "call that replaces its workspace");
    EXPECT(waited, "no workspace was replaced");
    stub::on_synchronize = nullptr;
}

// Products of very many rows or columns are launched, in grids that the runtime
// takes (below 2^32 threads): the stand-in refuses the others as it does.
static void grid_limits() {
    uint64_t outputs = 0;
    stub::on_launch = [&](const stub::Launch& l) {
        F32Launch f;
        if (!f32_launch(l.kernel, &f)) return;
        const auto g = l.arg<jh::F32Gemm>(0);
        outputs += (uint64_t)g.M * g.N;
        // the part of the product that a launch writes, and its operands' parts
        const int64_t at = g.C - fake(2), m0 = at / g.ldc, n0 = at % g.ldc;
        EXPECT(g.A - fake(0) == (g.ta ? m0 : m0 * g.lda) && g.B - fake(1) == (g.tb ? n0 * g.ldb : n0) &&
                   (!g.bias || g.bias - fake(3) == n0),
               "rows from %ld, columns from %ld: A + %ld, B + %ld", (long)m0, (long)n0, (long)(g.A - fake(0)),
               (long)(g.B - fake(1)));
    };
    const int kTop = INT32_MAX;
    for (int big : {1 << 22, (1 << 28) + 8, 1 << 29, (1 << 29) + 40, 1 << 30, kTop - 255}) {
        for (int small : {8, 16, 64, 200, 520}) {
            if ((int64_t)big * small > int64_t(1) << 37) continue;  // beyond a card's memory
            for (int K : {8, 64}) {
                EXPECT(jules_hip_gemm_bias_act(JH_BF16, JH_ACT_NONE, fake(0), fake(1), nullptr, fake(2), big, small, K,
                                               nullptr) == JH_OK,
                       "bf16 %d x %d x %d: %s", big, small, K, jules_hip_last_error());
                EXPECT(jules_hip_gemm_bias_act(JH_BF16, JH_ACT_NONE, fake(0), fake(1), nullptr, fake(2), small, big, K,
                                               nullptr) == JH_OK,
                       "bf16 %d x %d x %d: %s", small, big, K, jules_hip_last_error());
            }
            if (big % 16 == 0 && small % 16 == 0)
                EXPECT(jules_hip_matmul_int8(fake<int8_t>(0), fake<int8_t>(1), fake(2), big, small, 64, 1.0f, 1.0f,
                                             nullptr, nullptr) == JH_OK,
                       "int8 %d x %d: %s", big, small, jules_hip_last_error());
        }
        for (int n : {big, big + (big < kTop - 255 ? 0 : 255)})
            for (int small : {1, 3, 33, 100})
                for (int K : {1, 4, 64, 130}) {
                    if ((int64_t)n * std::max(small, K) > int64_t(1) << 37) continue;
                    outputs = 0;
                    EXPECT(jules_hip_gemm_bias_act(JH_F32, JH_ACT_RELU, fake(0), fake(1), fake(3), fake(2), n, small, K,
                                                   nullptr) == JH_OK,
                           "fp32 %d x %d x %d: %s", n, small, K, jules_hip_last_error());
                    EXPECT(jules_hip_gemm_bias_act(JH_F32, JH_ACT_RELU, fake(0), fake(1), fake(3), fake(2), small, n, K,
                                                   nullptr) == JH_OK,
                           "fp32 %d x %d x %d: %s", small, n, K, jules_hip_last_error());
                    EXPECT(outputs == 2 * (uint64_t)n * small, "%d x %d: %llu outputs", n, small,
                           (unsigned long long)outputs);
                    outputs = 0;
                    for (int t = 0; t < 4; ++t)
                        for (int flip : {0, 1}) {
                            const int M = flip ? small : n, N = flip ? n : small, ta = t & 1, tb = t >> 1;
                            EXPECT(jules_hip_sgemm(ta, tb, M, N, K, 1.0f, fake(0), ta ? M : K, fake(1), tb ? K : N, 1.0f,
                                                   fake(2), N, nullptr) == JH_OK,
                                   "sgemm %d x %d x %d ta=%d tb=%d: %s", M, N, K, ta, tb, jules_hip_last_error());
                        }
                    EXPECT(outputs == 8 * (uint64_t)n * small, "sgemm %d x %d: %llu outputs", n, small,
                           (unsigned long long)outputs);
                }
    }
}

// bf16 attention at a padded head dim reads its rows in place only where O lies
// apart from them (or is Q); any other overlap goes through copies.
static void overlapping_outputs() {
    bool in_place = false;
    stub::on_launch = [&](const stub::Launch& l) {
        in_place |= l.kernel.find("flash_fwd_bf16_pad") != std::string::npos;
    };
    const int64_t bytes = 1 * 2 * 100 * 80 * 2;
    for (int operand = 0; operand < 3; ++operand)
        for (int64_t off : {-bytes - 16, -bytes, -bytes + 16, int64_t(-160), int64_t(-16), int64_t(0), int64_t(16),
                            int64_t(160), bytes - 16, bytes, bytes + 16}) {
            in_place = false;
            EXPECT(jules_hip_flash_attn_fwd(JH_BF16, 0, 0.1f, fake(0), fake(1), fake(2), fake<char>(operand) + off,
                                            nullptr, 1, 2, 100, 80, nullptr) == JH_OK,
                   "%s", jules_hip_last_error());
            const bool sound = off <= -bytes || off >= bytes || (operand == 0 && off == 0);
            EXPECT(in_place == sound, "O at operand %d %+ld bytes", operand, (long)off);
        }
}

// The C++ training step and forward on host buffers: staged, launched, copied
// back and given back, at shapes with and without ranges of K, and after errors.
static void mlp_wrappers() {
    using namespace jules::kernel;
    int launches = 0;
    stub::on_launch = [&](const stub::Launch&) { ++launches; };
    const auto before = stub::allocations();
    {
        ExecutionArena arena;
        TilePlanner planner;
        const auto with_arena = stub::allocations();
        for (int M : {0, 1, 19, 64, 300})
            for (int K1 : {1, 23, 784})
                for (int N1 : {1, 17, 256})
                    for (int N2 : {1, 5, 10}) {
                        std::vector<float> X(M * K1), W1(K1 * N1), b1(N1), W2(N1 * N2), b2(N2), out(M * N2);
                        std::vector<float> dW1(K1 * N1), db1(N1), dW2(N1 * N2), db2(N2), dX(M * K1);
                        std::vector<int32_t> t(M);
                        for (float* dx : {dX.data(), (float*)nullptr}) {
                            launches = 0;
                            const auto r = interleavedMLPForwardBackward(
                                X.data(), W1.data(), b1.data(), W2.data(), b2.data(), t.data(), out.data(), dW1.data(),
                                db1.data(), dW2.data(), db2.data(), dx, M, K1, N1, N2, arena, planner);
                            EXPECT(lastStatus() == JH_OK && launches >= 5 && r.grads.dX == dx, "%d x %d x %d x %d: %s", M,
                                   K1, N1, N2, lastError());
                        }
                        const MLPParams p{W1.data(), b1.data(), W2.data(), b2.data(), M, K1, N1, N2};
                        fusedMLPForward(out.data(), X.data(), p, arena, planner);
                        EXPECT(lastStatus() == JH_OK, "%s", lastError());
                        const MLPParams bad{W1.data(), b1.data(), W2.data(), b2.data(), M, 0, N1, N2};
                        fusedMLPForward(out.data(), X.data(), bad, arena, planner);
                        EXPECT(lastStatus() == JH_ERR_SHAPE, "%d", lastStatus());
                    }
        EXPECT(stub::allocations() == with_arena, "%zu device buffers are left", stub::allocations().size());
    }
    EXPECT(stub::allocations() == before, "%zu device buffers are left", stub::allocations().size());
}

// Names what each product read from stdin launches: "f32 M N K", "bf16 M N K",
// "int8 M N K" or "sgemm ta tb M N K", one a line.  The fp32 tile as BM x BN x BK
// and its variant, with "folded" where it adds ranges of K itself; "whole" for
// the kernels of whole 256 x 256 tiles; "/3" for a ring of 3 stages; "split" where
// a reduction follows.
static void tiles() {
    std::string line, said;
    stub::on_launch = [&](const stub::Launch& l) {
        F32Launch f;
        int bm, bn, stages;
        const size_t cfg = l.kernel.find("TileCfg<");
        char s[80];
        if (f32_launch(l.kernel, &f))
            std::snprintf(s, sizeof s, "%dx%dx%d v%d%s", 2 * f.mt * f.mf, 2 * f.nt * f.mf, f.bk, f.v,
                          f.fold ? " folded" : "");
        else if (cfg != std::string::npos && std::sscanf(l.kernel.c_str() + cfg, "TileCfg<jh::%*[A-Za-z0-9], %d, %d, %*d, %*d, %*d, %*d, %d", &bm, &bn,
                                                         &stages) == 3)
            std::snprintf(s, sizeof s, stages == 3 ? "%dx%d/3" : "%dx%d", bm, bn);
        else if (l.kernel.find("_dma_kernel") != std::string::npos)
            std::snprintf(s, sizeof s, "whole");
        else if (l.kernel.find("_reduce_kernel") != std::string::npos)
            std::snprintf(s, sizeof s, " split");
        else
            std::snprintf(s, sizeof s, "%s", l.kernel.c_str());
        said += s;
    };
    while (std::getline(std::cin, line)) {
        std::istringstream in(line);
        std::string kind;
        int ta = 0, tb = 0, M = 0, N = 0, K = 0, st;
        in >> kind;
        if (kind == "sgemm") in >> ta >> tb;
        in >> M >> N >> K;
        said.clear();
        if (kind == "sgemm")
            st = jules_hip_sgemm(ta, tb, M, N, K, 1.0f, fake(0), ta ? M : K, fake(1), tb ? K : N, 1.0f, fake(2), N, nullptr);
        else if (kind == "int8")
            st = jules_hip_matmul_int8(fake<int8_t>(0), fake<int8_t>(1), fake(2), M, N, K, 1.0f, 1.0f, nullptr, nullptr);
        else
            st = jules_hip_gemm_bias_act(kind == "bf16" ? JH_BF16 : JH_F32, JH_ACT_NONE, fake(0), fake(1), nullptr,
                                         fake(2), M, N, K, nullptr);
        std::printf("%s: %s\n", line.c_str(), st == JH_OK ? said.c_str() : jules_hip_last_error());
    }
}

static const struct {
    const char* name;
    void (*run)();
} kChecks[] = {
    {"f32_offsets", f32_offsets},
    {"graph_workspace", graph_workspace},
    {"stream_locks", stream_locks},
    {"grid_limits", grid_limits},
    {"overlapping_outputs", overlapping_outputs},
    {"mlp_wrappers", mlp_wrappers},
    {"tiles", tiles},
};

int main(int argc, char** argv) {
    for (const auto& c : kChecks)
        if (argc == 2 && !std::strcmp(argv[1], c.name)) {
            c.run();
            stub::on_launch = nullptr;
            if (g_fail) std::fprintf(stderr, "%d failed expectations\n", g_fail);
            else std::printf("%s ok\n", c.name);
            return g_fail ? 1 : 0;
        }
    std::fprintf(stderr, "usage: host_launch <check>\n");
    return 2;
}
