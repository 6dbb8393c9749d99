"""The bf16 GEMM's tile kernel (gemm_tile.hpp) at the edges of its tiles, its K
slices and its K split, and the long-row kernel past its offset limit.

Tolerance: products of bf16 values are exact in fp32, a K-long fp32 sum is off
by at most K * 2^-24 of the sum of |terms| and the bf16 result by 2^-9 of
itself, so |y - ref| <= 2^-8 |ref| + 2^-20 sum |a b| holds with room for the
hardware exp2 of the activations."""
import pytest
import torch

from jules_amd import ops
from tests.helpers import case

pytestmark = pytest.mark.gpu


def _operands(dev, M, N, K, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    A = (torch.randn((M, K), generator=g, device=dev) / K ** 0.5).bfloat16()
    B = torch.randn((K, N), generator=g, device=dev).bfloat16()
    bias = torch.rand((N,), generator=g, device=dev) - 0.5
    return A, B, bias


def _check(y, A, B, bias, act):
    a, b = A.double(), B.double()
    z = a @ b
    z = z if bias is None else z + bias.double()
    ref = torch.nn.functional.silu(z) if act == "silu" else z
    bound = ref.abs() * 2.0 ** -8 + (a.abs() @ b.abs() + 1.0) * 2.0 ** -20
    assert ((y.double() - ref).abs() <= bound).all()


# the tile that each shape takes ("whole": the kernel of whole 256x256 tiles),
# and whether K is split; held by tests/test_tile_coverage.py
BF16_TILES = [
    (8, 8, 8, "32x64"), (8, 72, 16, "32x64"), (32, 64, 64, "32x64"), (40, 264, 136, "32x64"),
    (24, 504, 4352, "32x64 split"),
    (464, 1240, 80, "64x64"), (72, 1096, 4360, "64x64 split"),           # the last range is ragged
    (600, 2056, 1032, "64x128"), (1016, 384, 4544, "64x128 split"),
    (1272, 2304, 520, "128x128"), (536, 1968, 3736, "128x128 split"),
    (1000, 5000, 328, "128x256"), (512, 4224, 6984, "128x256 split"),
    (1288, 6152, 776, "256x256"), (1376, 3120, 4888, "256x256 split"),
    (3840, 2304, 32, "whole"), (3840, 2304, 96, "whole"), (3072, 3072, 160, "whole"),  # 1, 3 and 5 slices
    # whole tiles for half the chip and more, or a quarter and a short K: smaller
    # tiles took up to twice as long
    (1024, 4096, 512, "whole"), (2560, 2560, 256, "whole"), (2048, 4096, 1024, "whole"), (2304, 3840, 2560, "whole"),
]


@pytest.mark.parametrize("M,N,K,tile", BF16_TILES)
@pytest.mark.parametrize("act", ["none", "silu"])
def test_bf16_tiles(dev, M, N, K, tile, act):
    case(f"gemm bf16 tiles {M}x{N}x{K} {act}")
    A, B, bias = _operands(dev, M, N, K, M + N + K)
    bias = bias if act == "silu" else None
    y = ops.gemm_bias_act(A, B, bias, act)
    _check(y, A, B, bias, act)
    assert torch.equal(y, ops.gemm_bias_act(A, B, bias, act))


@pytest.mark.parametrize("M,N,K", [(8, 8, 1 << 22), (8, 1 << 24, 8)])
def test_bf16_long_rows(dev, M, N, K):
    case(f"gemm bf16 long rows {M}x{N}x{K}")
    A, B, _ = _operands(dev, M, N, K, 1)
    _check(ops.gemm_bias_act(A, B, None, "none"), A, B, None, "none")


def test_bf16_very_many_rows(dev):
    """2^30 rows: the smaller tiles would need more threads than a launch has."""
    case("gemm bf16 2^30 x 8 x 8")
    M, part = 1 << 30, 1 << 26
    A = torch.empty((M, 8), dtype=torch.bfloat16, device=dev)
    for i in range(0, M, part):
        A[i:i + part] = torch.rand((part, 1), device=dev) - 0.5
    B = torch.randn((8, 8), device=dev).bfloat16()
    y = ops.gemm_bias_act(A, B, None, "none")
    for i in range(0, M, part):
        _check(y[i:i + part], A[i:i + part], B, None, "none")


@pytest.mark.parametrize("K", [8, 40, 72, 4360])
def test_bf16_k_tail_keeps_rows_apart(dev, K):
    """An infinity in one row of A may not reach the row before it through
    the part of a K slice past the row's end."""
    case(f"gemm bf16 K tail {K}")
    A, B, _ = _operands(dev, 40, 136, K, 5)
    A[1::2] = float("inf")
    y = ops.gemm_bias_act(A, B, None, "none")
    _check(y[::2], A[::2].contiguous(), B, None, "none")
    assert not torch.isfinite(y[1::2]).any()


def test_bf16_split_under_capture(dev):
    """A shape whose K is split outside a graph: the captured call replays
    with the program's own calls in between."""
    case("gemm bf16 split under capture")
    A, B, bias = _operands(dev, 24, 504, 4352, 9)
    y = torch.empty((24, 504), dtype=torch.bfloat16, device=dev)
    s = torch.cuda.Stream()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        ops.gemm_bias_act(A, B, bias, "silu", out=y)
    for i in range(3):
        A.copy_((torch.randn(A.shape, device=dev) / 66).bfloat16())
        g.replay()
        eager = ops.gemm_bias_act(A, B, bias, "silu")
        torch.cuda.synchronize()
        _check(y, A, B, bias, "silu")
        _check(eager, A, B, bias, "silu")


@pytest.mark.parametrize("k", [1, 3])
def test_split_into_misaligned_outputs(dev, k):
    """Where K is split, an output that starts k elements past a 16-byte
    address holds the bits of an aligned one, and nothing around it is
    written."""
    case(f"split GEMMs into outputs off by {k}")

    def off(M, N, dtype):
        buf = torch.full((M * N + k + 8,), 7, dtype=dtype, device=dev)
        return buf, buf[k:k + M * N].view(M, N)

    A, B, bias = _operands(dev, 24, 504, 4352, 9)
    buf, out = off(24, 504, torch.bfloat16)
    assert torch.equal(ops.gemm_bias_act(A, B, bias, "silu", out=out), ops.gemm_bias_act(A, B, bias, "silu"))
    assert (buf[:k] == 7).all() and (buf[k + out.numel():] == 7).all()
    a8 = torch.randint(-128, 128, (72, 4368), device=dev, dtype=torch.int8)
    b8 = torch.randint(-128, 128, (4368, 1104), device=dev, dtype=torch.int8)
    buf, out = off(72, 1104, torch.float32)
    assert torch.equal(ops.matmul_int8(a8, b8, 0.5, 0.25, bias=None, out=out), ops.matmul_int8(a8, b8, 0.5, 0.25))
    assert (buf[:k] == 7).all() and (buf[k + out.numel():] == 7).all()


def test_split_leaves_a_graphs_workspace(dev):
    """A graph captured from a call that keeps the stream's workspace replays
    between eager GEMMs that split K on that stream."""
    case("gemm bf16 split on the stream of a captured int8 decode")
    g = torch.Generator(device=dev).manual_seed(2)
    a8 = torch.randint(-128, 128, (8, 1024), generator=g, device=dev, dtype=torch.int8)
    b8 = torch.randint(-128, 128, (1024, 512), generator=g, device=dev, dtype=torch.int8)
    one = torch.ones((), device=dev)
    A, B, _ = _operands(dev, 24, 4104, 4352, 11)
    y8 = torch.empty((8, 512), device=dev)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        ops.matmul_int8(a8, b8, 1.0, 1.0, out=y8)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            ops.matmul_int8(a8, b8, 1.0, 1.0, out=y8)
        for _ in range(3):
            y = ops.gemm_bias_act(A, B, None, "none")
            a8.copy_(torch.randint(-128, 128, a8.shape, generator=g, device=dev, dtype=torch.int8))
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(y8, _int8_ref(a8, b8, one, one, None))
            _check(y, A, B, None, "none")


def _int8_ref(A, B, rs, cs, bias):
    """The scalar path's arithmetic on the exact integer sums (each below
    2^31, so the float64 product holds it exactly)."""
    z = (A.double() @ B.double()).float() * (rs * cs)
    return z if bias is None else z + bias


INT8_TILES = [
    (23, 992, 2816, "32x64"), (22, 2832, 6720, "32x64 split"),
    (17, 16, 16, "64x64"), (40, 272, 144, "64x64"), (768, 1280, 320, "64x64"), (645, 688, 6768, "64x64"),
    (39, 2960, 8128, "64x64 split"), (72, 1104, 4368, "64x64 split"),    # the last range is ragged
    (222, 5264, 7328, "64x128"), (39, 5952, 6768, "64x128 split"),
    (540, 4112, 1040, "128x128"), (1000, 2064, 912, "128x128"),
    (796, 5616, 6864, "128x256"),
    (1304, 6160, 784, "128x256/3"), (1304, 6160, 2064, "256x256"),
    (2816, 3072, 128, "whole"), (2304, 3840, 320, "whole"),
    (768, 7168, 256, "whole"), (2048, 11520, 768, "whole"),
    # many tiles and a short K, 1 to 32 slices
    (33, 65552, 64, "128x256/3"), (2177, 4368, 80, "128x256/3"), (276, 24016, 144, "128x256/3"),
    (2281, 5376, 256, "128x256/3"), (2840, 6400, 2032, "128x256/3"),
]
# rows of any length: a kernel of their own
INT8_ROWS = [(1, 1, 1, ""), (3, 65, 17, ""), (64, 64, 64 - 1, ""), (65, 130, 129, ""), (33, 1000, 255, "")]


@pytest.mark.parametrize("M,N,K,tile", INT8_TILES + INT8_ROWS)
def test_int8_tiles(dev, M, N, K, tile):
    case(f"int8 tiles {M}x{N}x{K}")
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    A = torch.randint(-128, 128, (M, K), generator=g, device=dev, dtype=torch.int8)
    B = torch.randint(-128, 128, (K, N), generator=g, device=dev, dtype=torch.int8)
    sa = torch.rand((M,), generator=g, device=dev) + 0.01
    sb = torch.rand((N,), generator=g, device=dev) + 0.01
    bias = torch.rand((N,), generator=g, device=dev) - 0.5
    assert torch.equal(ops.matmul_w8a8(A, B, sa, sb, bias), _int8_ref(A, B, sa[:, None], sb, bias))
    f32 = torch.tensor(0.013, device=dev), torch.tensor(0.021, device=dev)
    assert torch.equal(ops.matmul_int8(A, B, 0.013, 0.021), _int8_ref(A, B, *f32, None))


def test_int8_misaligned_operands(dev):
    """Operands that start between 16-byte addresses, and end with their
    allocation's last byte."""
    case("int8 misaligned")
    M, N, K = 50, 96, 80
    buf = torch.randint(-128, 128, (M * K + K * N + 3,), device=dev, dtype=torch.int8)
    A, B = buf[3:3 + M * K].view(M, K), buf[3 + M * K:].view(K, N)
    one = torch.ones((), device=dev)
    assert torch.equal(ops.matmul_int8(A, B, 1.0, 1.0), _int8_ref(A, B, one, one, None))
