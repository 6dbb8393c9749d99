// flash_pad.hip - flash attention for head dims the kernels are not built
// for (1 <= D <= 128, D not 64 or 128), and the per-stream workspace shared
// by the entry points that take none.
//
// The reference's flashAttention (include/jules/Kernel/FlashAttention.h:
// 130-309) accepts any head_dim.  The MFMA kernels here are built for 64 and
// 128; other sizes are zero-padded to the next of the two, by the bf16 forward
// itself where rows are whole 16-byte pieces, else through the workspace.  Zero columns
// change neither the scores Q K^T, nor the log-sum-exp, nor the real columns
// of O (padded V columns only produce padded O columns), nor, in the
// backward, the real columns of dQ, dK and dV (rowsum(dO * O) is unchanged;
// the padded gradient columns come out as zeros).  The caller's scale is
// used as given (its default is 1/sqrt(D) of the real D).
#include <map>
#include <mutex>
#include <tuple>

#include "common.hpp"
#include "launch.hpp"

namespace jh {

namespace {
enum BufferUse { BUFFER_CALL, BUFFER_PARTIALS };

// A lock of its own: a call that waits for its stream to replace a buffer
// keeps no other stream's calls waiting.
struct StreamBuffer {
    std::recursive_mutex mu;
    void* ptr = nullptr;
    size_t bytes = 0;
};

hipError_t stream_buffer(BufferUse use, size_t need, hipStream_t s, void** ws, WorkspaceLock* lock) {
    static std::mutex mu;  // of the map only; its elements stay where they are
    static std::map<std::tuple<int, hipStream_t, BufferUse>, StreamBuffer> buffers;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    StreamBuffer* b;
    {
        std::lock_guard<std::mutex> map_lock(mu);
        b = &buffers[{dev, s, use}];
    }
    *lock = WorkspaceLock(b->mu);
    if (b->bytes < need) {
        if (b->ptr) {
            if ((e = hipStreamSynchronize(s)) != hipSuccess) return e;
            (void)hipFree(b->ptr);
        }
        b->ptr = nullptr;
        b->bytes = 0;
        if ((e = hipMalloc(&b->ptr, need)) != hipSuccess) {
            b->ptr = nullptr;
            return e;
        }
        b->bytes = need;
    }
    *ws = b->ptr;
    return hipSuccess;
}
}  // namespace

// One workspace per (device, stream), kept for the process: calls on one
// stream run in order and may share it, calls on other streams get their
// own.  A larger need replaces it once the stream is done with the old one.
// The lock is the caller's until it has enqueued every kernel that uses the
// workspace, so that threads sharing a stream neither interleave their kernels
// nor replace the buffer under each other; recursive, since a registry call
// holds it around entry points of the library.
hipError_t stream_workspace(size_t need, hipStream_t s, void** ws, WorkspaceLock* lock) {
    return stream_buffer(BUFFER_CALL, need, s, ws, lock);
}

// A graph captured after a warm-up holds the workspace's address.  A GEMM only
// splits K outside of captures, and with a buffer apart it neither writes nor
// replaces what such a graph replays into.
hipError_t stream_partials(hipStream_t s, void** ws, WorkspaceLock* lock) {
    return stream_buffer(BUFFER_PARTIALS, kMaxPartialBytes, s, ws, lock);
}

namespace {

// Up to 8 tensors, one per blockIdx.y, moved in pieces of T: 16 bytes where a
// row of D elements is whole pieces, else one element.
struct RowsArgs {
    void* dst[8];
    const void* src[8];
};
// dst[r][c] = c < n ? src[r][c] : 0 over [rows][1 << sh] (PAD), or
// dst[r][c] = src[r][c] for c < n, src rows 1 << sh wide
template <typename T, bool PAD>
__global__ void move_rows_kernel(RowsArgs a, int64_t rows, int n, int sh) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t r = i >> sh;
    const int c = (int)(i & ((1 << sh) - 1));
    if (r >= rows || (!PAD && c >= n)) return;
    T* d = static_cast<T*>(a.dst[blockIdx.y]);
    const T* s = static_cast<const T*>(a.src[blockIdx.y]);
    if (PAD) d[i] = c < n ? s[r * n + c] : T{};
    else d[r * n + c] = s[i];
}

inline size_t a256(size_t n) { return (n + 255) & ~size_t(255); }

// `count` tensors of `rows` rows, D elements of es bytes wide, into (PAD) or
// out of rows of Dp elements; one launch (a launch per tensor of 2-byte pieces
// took 4.2 us each at 2 x 16 x 333 x 80)
template <bool PAD>
hipError_t move_rows(const RowsArgs& a, int count, int64_t rows, int D, int Dp, size_t es, hipStream_t s) {
    auto go = [&](auto piece) {
        using T = decltype(piece);
        const int per = (int)(sizeof(T) / es), n = D / per;
        int sh = 0;
        while ((1 << sh) < Dp / per) ++sh;
        const int64_t total = rows << sh;
        hipLaunchKernelGGL((move_rows_kernel<T, PAD>), dim3((unsigned)((total + 255) / 256), (unsigned)count),
                           dim3(256), 0, s, a, rows, n, sh);
        return hipGetLastError();
    };
    if (D * es % 16 == 0) return go(u32x4_t{});
    return es == 2 ? go(uint16_t{}) : go(uint32_t{});
}

}  // namespace

int flash_padded_dim(int D) { return D <= 64 ? 64 : 128; }

hipError_t launch_flash_fwd_padded(int dtype, int causal, float scale, const void* Q, const void* K,
                                   const void* V, void* O, float* lse, int B, int H, int S, int D,
                                   hipStream_t s) {
    // the workspace holds copies of Q, K and V, so there O may lie over them;
    // without it O may be Q itself (a workgroup writes the rows that it alone
    // has read), but lies apart from Q otherwise and from K and V
    const auto apart = [&](const void* in) {
        const char *o = static_cast<const char*>(O), *i = static_cast<const char*>(in);
        const int64_t bytes = (int64_t)B * H * S * D * 2;
        return o + bytes <= i || i + bytes <= o;
    };
    if (flash_fwd_takes_rows(dtype, S, D) && (O == Q || apart(Q)) && apart(K) && apart(V))
        return launch_flash_fwd_rows(causal, scale, Q, K, V, O, lse, B, H, S, D, s);
    const int Dp = flash_padded_dim(D);
    const int64_t rows = (int64_t)B * H * S;
    const size_t es = dtype == JH_BF16 ? 2 : 4;
    const size_t one = a256((size_t)rows * Dp * es);
    void* ws = nullptr;
    WorkspaceLock lock;
    hipError_t e = stream_workspace(4 * one, s, &ws, &lock);
    if (e != hipSuccess) return e;
    char* w = static_cast<char*>(ws);
    if ((e = move_rows<true>({{w, w + one, w + 2 * one}, {Q, K, V}}, 3, rows, D, Dp, es, s))) return e;
    if ((e = launch_flash_fwd(dtype, causal, scale, w, w + one, w + 2 * one, w + 3 * one, lse, B, H, S, Dp, s)))
        return e;
    return move_rows<false>({{O}, {w + 3 * one}}, 1, rows, D, Dp, es, s);
}

hipError_t launch_flash_bwd_padded(int dtype, int causal, float scale, const void* Q, const void* K,
                                   const void* V, const void* O, const void* dO, const float* lse,
                                   void* dQ, void* dK, void* dV, int B, int H, int S, int D,
                                   void* bwd_ws, hipStream_t s) {
    const int Dp = flash_padded_dim(D);
    const int64_t rows = (int64_t)B * H * S;
    const size_t es = dtype == JH_BF16 ? 2 : 4;
    const size_t one = a256((size_t)rows * Dp * es);
    void* ws = nullptr;
    WorkspaceLock lock;
    hipError_t e = stream_workspace(8 * one, s, &ws, &lock);
    if (e != hipSuccess) return e;
    char* p[8];
    for (int i = 0; i < 8; ++i) p[i] = static_cast<char*>(ws) + i * one;  // Q K V O dO dQ dK dV
    if ((e = move_rows<true>({{p[0], p[1], p[2], p[3], p[4]}, {Q, K, V, O, dO}}, 5, rows, D, Dp, es, s))) return e;
    if ((e = launch_flash_bwd(dtype, causal, scale, p[0], p[1], p[2], p[3], p[4], lse, p[5], p[6], p[7],
                              B, H, S, Dp, bwd_ws, s)))
        return e;
    return move_rows<false>({{dQ, dK, dV}, {p[5], p[6], p[7]}}, 3, rows, D, Dp, es, s);
}

}  // namespace jh
