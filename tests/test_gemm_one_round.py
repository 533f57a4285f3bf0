"""fp16 products of one round of small tiles: those whose size does not divide a 256 x 256 block, the last ones of which lie against the edges
of M x N, and those whose two groups of waves share K tiles.  Which products take them, and whole numbers bit-exact (src/cutlass-gemm/gemm.cu:
277-294), also where D is C: what two tiles cover only one may store."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from _util import pkg

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cutlass-kernels_amd", "csrc")
SHIM = """#include "gemm_choice.h"
extern "C" int rows(int m, int n, int k, int batch, int *cols, int *tiles) {
  const cfk::GemmChoice c = cfk::choose_gemm_f16(m, n, k, batch);
  *cols = c.rows ? c.cols : c.tail_cols, *tiles = c.rows ? c.tiles : 0;
  return c.rows ? c.rows : c.tail_rows;
}
extern "C" int shared_from() { return cfk::kSharedFrom; }
"""
SHAPES = [  # L, M, N, tile
    (1, 256, 1280, (64, 32)), (2, 1024, 256, (64, 32)),
    (1, 1024, 1024 + 256, (96, 64)), (3, 512, 768, (96, 64)), (1, 256, 4608, (96, 64)),
    (1, 1536, 1536, (96, 96)), (1, 2304, 1024 + 256, (96, 128)), (1, 3072, 768, (96, 96)), (5, 256, 1792, (96, 128)), (1, 768, 4096, (96, 128)),
    (1, 2048, 2048, (128, 128)), (3, 1024, 1280, (128, 128)),
    (1, 3072, 1536, (128, 192)), (2, 2048, 1280, (192, 128)), (1, 512, 9472, (128, 192)), (1, 9216, 512, (192, 128)), (1, 5632, 1024, (192, 128)),
]


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("choice")
    (d / "shim.cpp").write_text(SHIM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", "-I", CSRC, "-o", str(d / "c.so"), str(d / "shim.cpp")], check=True)
    return ctypes.CDLL(str(d / "c.so"))


def _choice(lib, L, M, N, K):
    cols, tiles = ctypes.c_int(), ctypes.c_int()
    return (lib.rows(M, N, K, L, ctypes.byref(cols), ctypes.byref(tiles)), cols.value), tiles.value


def test_rule_without_gpu(lib):
    for L, M, N, tile in SHAPES:
        for K in (512, 1088, 8192):
            got, tiles = _choice(lib, L, M, N, K)
            assert got == tile, (L, M, N, K, got)
            if tiles: assert tiles == L * -(-M // tile[0]) * -(-N // tile[1]) <= 256
    # all of them at once on the CUs, or a size that divides a block
    for M in range(256, 4097, 256):
        for N in range(256, 4097, 256):
            for L in (1, 2, 5):
                if L * M * N <= 128 * 65536:
                    (rows, cols), tiles = _choice(lib, L, M, N, 1024)
                    assert tiles <= 256 and (tiles or (256 % rows == 0 and 256 % cols == 0 and L * M * N <= 256 * rows * cols * 4))
    assert lib.shared_from() == 1088   # (the sizes of K below are on either side)


# K tiles of 64: as few as the rule takes, an odd number; the first length of the shared form, odd and even with a refill of all its five stages
@pytest.mark.gpu
@pytest.mark.parametrize("K", [512, 576, 1024, 1088, 1152])
@pytest.mark.parametrize("layout", [0, 1])
def test_whole_numbers_bit_exact(K, layout):
    import torch
    gen = torch.Generator("cuda").manual_seed(K + layout)
    draw = lambda *shape: torch.randint(-4, 5, shape, generator=gen, device="cuda").float()
    for L, M, N, tile in SHAPES:
        a, b, c = draw(L, M, K), draw(L, N, K), draw(L, M, N)
        bt = b if layout == 0 else b.transpose(1, 2).contiguous()
        ab = torch.stack([torch.mm(a[i], b[i].t().contiguous()) for i in range(L)])   # (below 2^15: exact in fp32 in any order)
        h = [x.half().contiguous() for x in (a, bt, c)]
        for alpha, beta, c_in, out in [(0.5, 0.0, None, None), (0.5, -2.0, h[2], None), (1.0, 1.0, h[2].clone(), "c")]:
            got = pkg.gemm(h[0], h[1], c=c_in, alpha=alpha, beta=beta, out=c_in if out else None, layout=layout)
            torch.cuda.synchronize()
            assert torch.equal(got, (alpha * ab + beta * c).half()), (L, M, N, K, tile, alpha, beta)
    print(f"K={K} layout {layout}: {len(SHAPES)} products", flush=True)
