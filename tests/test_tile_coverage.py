"""The shapes that the GPU tests of the GEMM tiles name a tile for do take that
tile: what each of them launches, from tests/cpp/host_launch, without a GPU."""
import os
import subprocess

import pytest

from tests.test_gpu_gemm import F32_TILES
from tests.test_gpu_gemm_tiles import BF16_TILES, INT8_TILES
from tests.test_gpu_sgemm import SGEMM_TILES
from tests.test_host_launch import _binary


@pytest.mark.parametrize("kind,shapes", [("f32", F32_TILES), ("bf16", BF16_TILES), ("int8", INT8_TILES),
                                         ("sgemm", SGEMM_TILES)])
def test_shapes_take_their_tiles(kind, shapes):
    if subprocess.run(["g++", "--version"], capture_output=True).returncode != 0:
        pytest.skip("no g++")
    want = [(" ".join([kind, *map(str, s[:-1])]), s[-1]) for s in shapes]
    r = subprocess.run([_binary(), "tiles"], input="".join(f"{q}\n" for q, _ in want), capture_output=True, text=True,
                       env=dict(os.environ, ASAN_OPTIONS="detect_leaks=0"), timeout=120)
    assert r.returncode == 0, r.stderr[-2000:]
    assert r.stdout.splitlines()[:len(want)] == [f"{q}: {tile}" for q, tile in want]
