"""fp32 products in tiles of 64 x 64 and 32 x 32 side by side (gemm_kernel_f32_mix): which products take them, whole numbers bit-exact at the edges
of the rule, and the error against float64, which depends on how many partial sums an element has."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

import oracle
from _util import pkg, to_dev

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cutlass-kernels_amd", "csrc")
SHIM = """#include "gemm_choice.h"
extern "C" int mix(int blocks, int k) { const cfk::GemmMix m = cfk::choose_gemm_f32_mix(blocks, k); return m.sums ? m.blocks64 * 8 + m.sums : -1; }
extern "C" int edge(int blocks) { return cfk::choose_gemm_f32(blocks); }
"""


def test_rule_without_gpu(tmp_path):
    (tmp_path / "shim.cpp").write_text(SHIM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", "-I", CSRC, "-o", str(tmp_path / "c.so"), str(tmp_path / "shim.cpp")], check=True)
    lib = ctypes.CDLL(str(tmp_path / "c.so"))
    for blocks in range(1, 1100):
        for K in (64, 1024, 4096):
            m = lib.mix(blocks, K)
            if m < 0: continue
            # whole rounds of 64 x 64 tiles, at most 12 blocks behind them, and as many partial sums as in the one tile size
            assert m // 8 == blocks // 16 * 16 * (blocks > 16) and blocks - m // 8 <= 12
            assert m % 8 == {128: 1, 64: 2, 32: 4}[lib.edge(blocks)]
    assert lib.mix(36, 1536) == 32 * 8 + 4 and lib.mix(10, 512) == 4 and lib.mix(10, 2048) == -1
    for blocks in (1, 8, 13, 16, 29, 31, 32, 48, 64, 128, 1024): assert lib.mix(blocks, 1024) == -1


# 4 sums: one block behind a round, 9 and 12 blocks without one, a batch; 2 sums: 76 blocks; 1 sum: 54
@pytest.mark.gpu
@pytest.mark.parametrize("L,M,N,K", [(1, 4352, 256, 64), (1, 768, 768, 64), (3, 1024, 256, 192), (4, 256, 1280, 320), (3, 1024, 768, 128), (1, 4864, 1024, 64), (2, 2304, 768, 64)])
@pytest.mark.parametrize("beta", [0.0, -3.0])
def test_whole_numbers_bit_exact(L, M, N, K, beta):
    rng = np.random.default_rng(L * 1000 + M + N + K)
    a, b, c = (rng.integers(-3, 4, s).astype(np.float32) for s in ((L, M, K), (L, N, K), (L, M, N)))
    got = pkg.gemm(to_dev(a), to_dev(b), c=to_dev(c) if beta else None, alpha=2.0, beta=beta).cpu().numpy()
    for i in range(L):
        assert np.array_equal(got[i], 2.0 * oracle.gemm_f32(a[i], b[i]) + beta * c[i])


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,limit", [(1280, 1024, 2048, 5e-7), (4864, 1024, 1024, 5e-7), (3456, 1024, 1024, 7e-7)])
def test_error_against_float64(M, N, K, limit):
    """Half a unit of the last place per addition in a random walk: 2^-24 sqrt(K / (3 sums)) of the size of the result, 1.0 to 1.3 of which the kernels with
    one tile size show (1024 of K: 2 sums 4.1e-7, 1 sum 5.7e-7; 2048, 4 sums 4.1e-7)."""
    import torch
    torch.manual_seed(3)
    M = M // 256 * 256
    a, b = (torch.rand(s, device="cuda:0") * 2 - 1 for s in ((M, K), (N, K)))
    want = a.double() @ b.double().T
    got = pkg.gemm(a, b).double()
    assert float((got - want).norm() / want.norm()) <= limit
