"""Which macro tiles cfk_gemm runs a shape in (cutlass-kernels_amd/csrc/gemm_choice.h, host code): the shapes of test_gemm.py take the
kernels that they are there for, and near ties do not go to a tile that was measured to be the slower one."""
import ctypes
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cutlass-kernels_amd", "csrc")
SHIM = """#include "gemm_choice.h"
extern "C" void f16(int m, int n, int k, int batch, int *out) {
  const cfk::GemmChoice c = cfk::choose_gemm_f16(m, n, k, batch);
  const int v[] = {c.rows, c.cols, c.tiles, c.tail_rows, c.tail_cols, c.tail_blocks};
  for (int i = 0; i < 6; ++i) out[i] = v[i];
}
extern "C" int f32(int blocks) { return cfk::choose_gemm_f32(blocks); }
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("choice")
    (d / "shim.cpp").write_text(SHIM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-fsanitize=undefined", "-fno-sanitize-recover", "-shared", "-fPIC", "-I", CSRC,
                    "-o", str(d / "choice.so"), str(d / "shim.cpp")], check=True)
    return ctypes.CDLL(str(d / "choice.so"))


def _f16(lib, L, M, N, K):
    out = (ctypes.c_int * 6)()
    lib.f16(M, N, K, L, out)
    return tuple(out)


BLOCKS = (256, 256)


@pytest.mark.parametrize("L,M,N,first,tail", [
    # test_macro_tiles_integer_inputs_bit_exact, test_main_loop_of_every_tile_size_bit_exact
    (1, 256, 256, None, (32, 32)), (1, 512, 512, None, (32, 32)), (1, 256, 1280, None, (64, 64)), (1, 1024, 1024, None, (64, 64)),
    (17, 256, 256, None, (128, 64)), (1, 1024, 2048, None, (128, 64)), (2, 1024, 1024, None, (128, 64)), (1, 256, 8448, None, (128, 128)),
    (4, 1024, 1024, None, (128, 128)), (1, 2048, 2048, None, (128, 128)), (65, 256, 256, None, (256, 128)), (1, 4096, 2048, None, (256, 128)),
    (129, 256, 256, BLOCKS, None), (257, 256, 256, BLOCKS, (32, 32)),
    # test_tiles_behind_a_whole_round_bit_exact
    (264, 256, 256, BLOCKS, (64, 64)), (280, 256, 256, BLOCKS, (128, 64)), (310, 256, 256, BLOCKS, (128, 128)), (384, 256, 256, BLOCKS, (256, 128)),
    # test_last_round_in_tiles_bit_exact
    (1, 6144, 4096, (192, 256), None),
    # test_macro_tiles_beyond_half_a_round_bit_exact, test_macro_tiles_at_an_edge_without_c_bit_exact
    (1, 3072, 3072, (192, 192), None), (2, 1280, 3328, (192, 192), None), (1, 3072, 4096, (192, 256), None), (1, 1280, 7168, (192, 256), None),
    (1, 4096, 3072, BLOCKS, None), (1, 1792, 5888, (192, 256), None),
    (1, 2560, 6656, (320, 256), None), (1, 2816, 6144, (320, 256), None),
    # test_c_of_64_mb_and_more_bit_exact
    (1, 8192, 8192, BLOCKS, None), (2, 4352, 4096, (320, 256), None)])
@pytest.mark.parametrize("K", [64, 192, 448])
def test_shapes_take_the_tiles_they_test(lib, L, M, N, first, tail, K):
    rows, cols, tiles, trows, tcols, tblocks = _f16(lib, L, M, N, K)
    assert (rows, cols) == (first or (0, 0)) and (trows, tcols) == (tail or (0, 0))
    covered = tiles if first in (None, BLOCKS) else L * (M // 256) * (N // 256)
    assert covered + tblocks == L * (M // 256) * (N // 256)
    if first not in (None, BLOCKS): assert tiles == L * -(-M // rows) * -(-N // cols) and tblocks == 0


@pytest.mark.parametrize("L,M,N,K", [
    (7, 1024, 5120, 640),      # 60 us in blocks and small tiles, 76 in 256 x 192 tiles
    (6, 512, 7168, 1024), (6, 1024, 5888, 832), (6, 1024, 3584, 1216), (6, 1024, 3584, 2112), (6, 512, 7680, 384),
    (3, 1024, 7424, 256),
    (8, 768, 3072, 704), (8, 768, 3072, 1792), (4, 768, 6144, 1856)])   # ... and 192 x 192: 76 and 79 us, 79 and 84
def test_near_ties_stay_in_blocks(lib, L, M, N, K):
    assert _f16(lib, L, M, N, K)[:2] == BLOCKS


@pytest.mark.parametrize("K", [1664, 2112, 4096, 8192])
@pytest.mark.parametrize("L,M,N,tiles", [(1, 4096, 3072, 256), (5, 256, 7168, 190)])
def test_256_x_192_where_it_is_the_faster_one(lib, L, M, N, tiles, K):
    # (test_256_x_192_tiles_bit_exact; 256 tiles in one round against 192 blocks: 83 against 87 us at K=4096)
    assert _f16(lib, L, M, N, K) == (256, 192, tiles, 0, 0, 0)


def test_limits(lib):
    # 320 rows of a K-contiguous operand have to stay within 32-bit byte offsets, like the 256 of a block
    k = (1 << 32) // (320 * 2) // 64 * 64
    assert 320 * k * 2 >= 1 << 32 or _f16(lib, 1, 2560, 6656, k)[:2] == (320, 256)
    assert _f16(lib, 1, 2560, 6656, k + 64)[:2] == BLOCKS
    # fewer rows than a tile has: 256 rows run in no 320-row tile
    assert all(_f16(lib, L, 256, 256, 64)[0] in (0, 256) for L in range(1, 1500))
    # every block is covered once, by the batch's order of blocks
    for blocks in range(1, 1500):
        rows, cols, tiles, _, _, tail = _f16(lib, blocks, 256, 256, 512)
        if (rows, cols) in ((0, 0), BLOCKS): assert tiles + tail == blocks


@pytest.mark.parametrize("blocks,edge", [(1, 32), (36, 32), (257, 64), (400, 64), (1024, 128)])
def test_fp32_tiles(lib, blocks, edge):
    assert lib.f32(blocks) == edge
