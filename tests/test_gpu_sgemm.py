"""jules_hip_sgemm on strided operands against fp64.

Tolerance: each output is one fma chain over K, or a few chains added, in fp32,
so it is off by at most K * 2^-24 of the sum of its |terms|; alpha and beta add
two roundings of the result."""
import pytest
import torch

from jules_amd import _lib
from tests.helpers import case

pytestmark = pytest.mark.gpu


def _strided(dev, rows, cols, ld, g):
    """rows x cols values in rows of ld floats, the rest of them as allocated."""
    m = torch.empty((rows, ld), device=dev)[:, :cols]
    m.copy_(torch.rand((rows, cols), generator=g, device=dev) * 2 - 1)
    return m


def _check_sgemm(dev, ta, tb, M, N, K, lda=None, ldb=None, ldc=None, alpha=1.0, beta=0.0):
    case(f"sgemm ta={ta} tb={tb} {M}x{N}x{K} lda={lda} ldb={ldb} ldc={ldc} alpha={alpha} beta={beta}")
    g = torch.Generator(device=dev).manual_seed(M + 3 * N + 5 * K)
    ar, ac = (K, M) if ta else (M, K)
    br, bc = (N, K) if tb else (K, N)
    A, B = _strided(dev, ar, ac, lda or ac, g), _strided(dev, br, bc, ldb or bc, g)
    C = _strided(dev, M, N, ldc or N, g)
    a, b, c = (A.T if ta else A).double(), (B.T if tb else B).double(), C.double()
    st = _lib.lib().jules_hip_sgemm(ta, tb, M, N, K, alpha, A.data_ptr(), A.stride(0), B.data_ptr(), B.stride(0), beta,
                                    C.data_ptr(), C.stride(0), torch.cuda.current_stream().cuda_stream)
    assert st == 0, _lib.lib().jules_hip_last_error()
    ref = alpha * (a @ b) + beta * c
    terms = abs(alpha) * (a.abs() @ b.abs()) + abs(beta) * c.abs()
    assert ((C.double() - ref).abs() <= (K + 2) * 2.0 ** -24 * terms).all()


@pytest.mark.parametrize("ta,tb,M,N", [(0, 0, 1, (1 << 29) + 40), (1, 0, (1 << 29) + 41, 1), (0, 1, 1, (1 << 29) + 3)])
def test_more_tiles_than_a_launch_has(dev, ta, tb, M, N):
    _check_sgemm(dev, ta, tb, M, N, 3, alpha=0.5, beta=-1.0)


@pytest.mark.parametrize("ta,tb,M,N,K,lda,ldb", [
    # slices that span 2^32 bytes of an operand: 64-bit offsets within a tile
    (0, 0, 33, 40, 70, 70, 17_200_000), (1, 0, 33, 40, 70, 17_200_000, 40),
    (0, 1, 33, 33, 70, 70, 34_700_000), (1, 1, 40, 33, 70, 17_200_000, 70),
    # those that only the deepest slice (128 k) would span
    (0, 0, 32, 32, 256, 256, 9_000_000), (1, 0, 32, 32, 256, 9_000_000, 32),
    # fewer k than a slice has
    (0, 0, 5, 32, 10, 10, 20_000_000), (1, 1, 32, 5, 3, 80_000_000, 3),
])
def test_wide_leading_dimensions(dev, ta, tb, M, N, K, lda, ldb):
    _check_sgemm(dev, ta, tb, M, N, K, lda, ldb)


# every tile of each orientation (a transposed B has none of 128x128), with
# 16-byte and 4-byte loads where an operand's k is the outer dimension; held by
# tests/test_tile_coverage.py
SGEMM_TILES = [
    (0, 0, 41, 45, 19, "32x32x64 v1"), (0, 0, 1001, 1021, 35, "64x64x32 v1"), (0, 0, 1024, 2048, 20, "64x128x16 v4"),
    (0, 0, 2040, 4092, 72, "128x128x16 v4"), (0, 0, 2041, 4089, 69, "128x128x16 v1"),
    (0, 0, 70, 50, 700, "32x32x64 v1 split"),
    (0, 0, 190, 230, 270, "32x32x128 v1 folded"), (0, 0, 130, 260, 2050, "64x128x16 v4 split"),
    (1, 0, 33, 48, 65, "32x32x64 v1"), (1, 0, 1024, 1008, 36, "64x64x32 v4"), (1, 0, 1001, 1021, 35, "64x64x32 v1"),
    (1, 0, 1024, 2048, 20, "64x128x16 v4"), (1, 0, 1001, 2041, 21, "64x128x16 v1"),
    (1, 0, 2040, 4092, 72, "128x128x16 v4"), (1, 0, 2041, 4089, 69, "128x128x16 v1"),
    (1, 0, 70, 50, 700, "32x32x64 v1 split"),
    (1, 0, 190, 230, 270, "32x32x128 v1 folded"), (1, 0, 300, 300, 300, "32x32x128 v4 folded"),
    (1, 0, 130, 260, 2050, "64x128x16 v1 split"),
    (0, 1, 33, 48, 65, "32x32x64 v4"), (0, 1, 1001, 1021, 35, "64x64x32 v4"), (0, 1, 1001, 2041, 21, "64x128x16 v4"),
    (0, 1, 2041, 4089, 69, "64x128x16 v4"), (0, 1, 70, 50, 700, "32x32x64 v4 split"),
    (0, 1, 190, 230, 270, "32x32x128 v4 folded"),
    (0, 1, 130, 260, 2050, "64x128x16 v4 split"),
    (1, 1, 33, 48, 65, "32x32x64 v1"), (1, 1, 1024, 1008, 36, "64x64x32 v4"), (1, 1, 1001, 1021, 35, "64x64x32 v1"),
    (1, 1, 1024, 2048, 20, "64x128x16 v4"), (1, 1, 1001, 2041, 21, "64x128x16 v1"),
    (1, 1, 70, 50, 700, "32x32x64 v1 split"),
    (1, 1, 190, 230, 270, "32x32x128 v1 folded"), (1, 1, 300, 300, 300, "32x32x128 v4 folded"),
    (1, 1, 130, 260, 2050, "64x128x16 v1 split"), (1, 1, 64, 64, 4096, "32x32x64 v4 split"),
]


@pytest.mark.parametrize("ta,tb,M,N,K,tile", SGEMM_TILES)
def test_sgemm_tiles(dev, ta, tb, M, N, K, tile):
    """Padded leading dimensions, alpha and beta."""
    ar, br = (M if ta else K) + 3, (K if tb else N) + 5
    _check_sgemm(dev, ta, tb, M, N, K, ar, br, N + 2, alpha=0.75, beta=-1.25)
