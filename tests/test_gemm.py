"""GPU parity of the dense GEMM (secondary bench, same tile engine) against the CPU oracle.
The reference checks its GEMM examples by equality on integer-valued inputs
(src/cutlass-gemm/gemm.cu:277-294, 329-359; src/cute-gemm-tma-gma/gemm.cu:645-651); so does this."""
import numpy as np
import pytest

import oracle
from _util import pkg, to_dev

pytestmark = pytest.mark.gpu


def _run(a, b, layout):
    import torch
    c = pkg.gemm_f16(to_dev(a.astype(np.float16)), to_dev(b.astype(np.float16)), layout=layout)
    torch.cuda.synchronize()
    return c.cpu().numpy()


@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("M,N,K", [(256, 256, 64), (512, 768, 320), (1024, 256, 1024)])
def test_integer_inputs_bit_exact(M, N, K, layout):
    rng = np.random.default_rng(M + N + K)
    a = rng.integers(-8, 9, (M, K)).astype(np.float32)
    b = rng.integers(-8, 9, (N, K)).astype(np.float32)       # logical B^T: b[n, k]
    want = oracle.gemm_f32(a, b).astype(np.float16)           # exact fp32 sums, one RNE rounding to fp16
    got = _run(a, b if layout == 0 else np.ascontiguousarray(b.T), layout)
    assert np.array_equal(got.view(np.uint16), want.view(np.uint16))


@pytest.mark.parametrize("layout", [0, 1])
def test_uniform_inputs(layout):
    M, N, K = 512, 512, 2048
    a = pkg.testbed.uniform((M, K), 1).astype(np.float16)
    b = pkg.testbed.uniform((N, K), 2).astype(np.float16)
    want = oracle.gemm_f32(a.astype(np.float32), b.astype(np.float32))
    got = _run(a, b if layout == 0 else np.ascontiguousarray(b.T), layout).astype(np.float32)
    # fp32 accumulation in a different order + one fp16 rounding of |c| <~ 60
    np.testing.assert_allclose(got, want, rtol=2e-3, atol=2e-3)


def test_config5_row_sample():
    # benchmark configuration 5: M=N=K=8192, U(-1,1) fp16, fp32 accumulate, fp16 C; 24 sampled rows against the oracle
    import torch
    M = N = K = 8192
    a = pkg.testbed.uniform((M, K), 3).astype(np.float16)
    b = pkg.testbed.uniform((N, K), 4).astype(np.float16)
    c = pkg.gemm_f16(to_dev(a), to_dev(b))
    torch.cuda.synchronize()
    rows = np.sort(np.random.default_rng(9).choice(M, 24, replace=False)).astype(np.int32)
    rows[0], rows[-1] = 0, M - 1
    want = oracle.gemm_f32(a.astype(np.float32), b.astype(np.float32), rows=rows)
    got = c[torch.from_numpy(rows).long().cuda()].float().cpu().numpy()
    np.testing.assert_allclose(got, want, rtol=2e-3, atol=1e-2)


@pytest.mark.parametrize("dtype", [np.float16, np.float32])
def test_alpha_beta_batch_integer_inputs_bit_exact(dtype):
    # the CUTLASS-API example's run: D = alpha * A.B + beta * C on integer-valued operands in [-8, 8], checked for
    # EQUALITY (src/cutlass-gemm/gemm.cu:277-294, 318-359); plus the CuTe example's batch count L (gemm.cu:519-521).
    # Everything is an integer below 2^24 in fp32, so alpha = 2, beta = -3 keep the result exact before the final
    # rounding to the output type.
    import torch
    L, M, N, K = 3, 256, 512, 192
    rng = np.random.default_rng(17)
    a = rng.integers(-8, 9, (L, M, K)).astype(np.float32)
    b = rng.integers(-8, 9, (L, N, K)).astype(np.float32)
    c = rng.integers(-8, 9, (L, M, N)).astype(np.float32)
    want = np.stack([2.0 * oracle.gemm_f32(a[i], b[i]) - 3.0 * c[i] for i in range(L)]).astype(dtype)
    got = pkg.gemm(to_dev(a.astype(dtype)), to_dev(b.astype(dtype)), c=to_dev(c.astype(dtype)), alpha=2.0, beta=-3.0)
    torch.cuda.synchronize()
    assert np.array_equal(got.cpu().numpy(), want)
    # beta = 0 must not read C (NaNs there would otherwise leak), and D may alias C
    cn = to_dev(np.full((L, M, N), np.nan, dtype))
    got = pkg.gemm(to_dev(a.astype(dtype)), to_dev(b.astype(dtype)), c=cn, alpha=1.0, beta=0.0, out=cn)
    torch.cuda.synchronize()
    assert np.array_equal(got.cpu().numpy(), np.stack([oracle.gemm_f32(a[i], b[i]) for i in range(L)]).astype(dtype))


@pytest.mark.parametrize("K", [64, 192, 320])
@pytest.mark.parametrize("dtype,layout", [(np.float16, 0), (np.float16, 1), (np.float32, 0)])
@pytest.mark.parametrize("L,M,N", [
    (1, 256, 256), (1, 512, 512), (1, 256, 1280), (1, 1024, 1024), (17, 256, 256), (2, 1024, 1024), (1, 256, 8448),
    (4, 1024, 1024), (65, 256, 256), (1, 4096, 2048), (129, 256, 256), (257, 256, 256)])
def test_macro_tiles_integer_inputs_bit_exact(L, M, N, K, dtype, layout):
    # 1 to 257 blocks of 256 x 256 on either side of every line where the macro tile changes (4, 16, 32, 64, 128 blocks, and
    # one block beyond a whole round of the CUs), with fewer K tiles than wave groups, a last turn that not all groups have
    # a tile for, and whole turns.  Integers: every sum is exact in fp32 in any order.
    import torch
    rng = np.random.default_rng(L + M + N + K)
    a = rng.integers(-8, 9, (L, M, K)).astype(np.float32)
    b = rng.integers(-8, 9, (L, N, K)).astype(np.float32)
    c = rng.integers(-8, 9, (L, M, N)).astype(np.float32)
    bt = b if layout == 0 else np.ascontiguousarray(b.transpose(0, 2, 1))
    got = pkg.gemm(to_dev(a.astype(dtype)), to_dev(bt.astype(dtype)), c=to_dev(c.astype(dtype)), alpha=0.5, beta=-1.0, layout=layout)
    torch.cuda.synchronize()
    got = got.cpu().numpy()
    for i in sorted({0, L // 2, L - 1}):
        want = (0.5 * oracle.gemm_f32(a[i], b[i]) - c[i]).astype(dtype)
        assert np.array_equal(got[i], want), i


@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("M,N", [(512, 512), (1024, 1024), (1024, 2048), (2048, 2048), (4096, 2048)])
def test_main_loop_of_every_tile_size_bit_exact(M, N, layout):
    # 33 K tiles of 64, one, two or four of them per turn and two to four turns in the LDS: every tile size (32 x 32, 64 x 64, 128 x 64,
    # 128 x 128, 256 x 128) refills each of its slots more than once while others multiply, and the last turn has a tile for one wave
    # group only
    import torch
    K = 2112
    rng = np.random.default_rng(M + N)
    a = rng.integers(-8, 9, (M, K)).astype(np.float32)
    b = rng.integers(-8, 9, (N, K)).astype(np.float32)
    want = oracle.gemm_f32(a, b).astype(np.float16)
    got = pkg.gemm(to_dev(a.astype(np.float16)), to_dev((b if layout == 0 else np.ascontiguousarray(b.T)).astype(np.float16)), layout=layout)
    torch.cuda.synchronize()
    assert np.array_equal(got.cpu().numpy(), want)


@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("K", [192, 256])
def test_last_round_in_tiles_bit_exact(K, layout):
    # 384 blocks of 256 x 256, which run as 512 tiles of 192 x 256: two whole rounds of the CUs
    import torch
    M, N = 6144, 4096
    rng = np.random.default_rng(K)
    a = rng.integers(-8, 9, (M, K)).astype(np.float32)
    b = rng.integers(-8, 9, (N, K)).astype(np.float32)
    got = pkg.gemm(to_dev(a.astype(np.float16)), to_dev((b if layout == 0 else np.ascontiguousarray(b.T)).astype(np.float16)), layout=layout)
    torch.cuda.synchronize()
    rows = np.arange(3, M, 61, dtype=np.int32)      # four of every row of blocks
    want = oracle.gemm_f32(a, b, rows=rows).astype(np.float16)
    assert np.array_equal(got.cpu().numpy()[rows], want)


@pytest.mark.parametrize("with_c", [False, True])
@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("L", [264, 280, 310, 384])
@pytest.mark.parametrize("K", [192, 256])
def test_tiles_behind_a_whole_round_bit_exact(L, K, layout, with_c):
    # the 8, 24, 54 and 128 blocks behind the first round of the CUs are tiles of 64 x 64, 128 x 64, 128 x 128 and 256 x 128
    # (test_gemm_choice.py asks for that), with as many K tiles as the largest has stages and one more
    import torch
    gen = torch.Generator(device="cuda").manual_seed(L + K)
    a, b, c = (torch.randint(-8, 9, shape, generator=gen, device="cuda").half() for shape in ((L, 256, K), (L, 256, K), (L, 256, 256)))
    kw = dict(c=c, alpha=0.5, beta=-1.0) if with_c else {}
    got = pkg.gemm(a, b if layout == 0 else b.transpose(1, 2).contiguous(), layout=layout, **kw)
    torch.cuda.synchronize()
    for i in (0, 255, 256, 257, (256 + L) // 2, L - 1):
        want = oracle.gemm_f32(a[i].float().cpu().numpy(), b[i].float().cpu().numpy())
        if with_c: want = 0.5 * want - c[i].float().cpu().numpy()
        assert np.array_equal(got[i].cpu().numpy(), want.astype(np.float16)), i


@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("L,M,N", [
    (1, 3072, 3072),     # 192 x 192 tiles, 256 of them
    (2, 1280, 3328),     # ... the last ones of two problems against both edges
    (1, 3072, 4096),     # 192 x 256
    (1, 1280, 7168),     # ... the last row of tiles against the edge
    (1, 4096, 3072),     # 256 x 256
    (1, 1792, 5888),     # 192 x 256, the last row of tiles against the edge
    (1, 2560, 6656),     # 320 x 256
    (1, 2816, 6144)])    # ... the last row of tiles against the edge
@pytest.mark.parametrize("K", [64, 192, 448])
def test_macro_tiles_beyond_half_a_round_bit_exact(L, M, N, K, layout):
    # one, three and seven K tiles; D over C: what two tiles at an edge both cover is read and stored once
    import torch
    rng = np.random.default_rng(M + N + K)
    a = rng.integers(-8, 9, (L, M, K)).astype(np.float32)
    b = rng.integers(-8, 9, (L, N, K)).astype(np.float32)
    c = rng.integers(-8, 9, (L, M, N)).astype(np.float32)
    bt = b if layout == 0 else np.ascontiguousarray(b.transpose(0, 2, 1))
    d = to_dev(c.astype(np.float16))
    pkg.gemm(to_dev(a.astype(np.float16)), to_dev(bt.astype(np.float16)), c=d, alpha=0.5, beta=-1.0, layout=layout, out=d)
    torch.cuda.synchronize()
    rows = np.unique(np.concatenate([np.arange(3, M, 61), np.arange(M - 70, M)])).astype(np.int32)
    got = d.cpu().numpy()
    for i in range(L):
        want = (0.5 * oracle.gemm_f32(a[i], b[i], rows=rows) - c[i][rows]).astype(np.float16)
        assert np.array_equal(got[i][rows], want), i


@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("L,M,N", [
    (1, 8192, 8192),     # 256 x 256 blocks, 134 MB of C
    (2, 4352, 4096)])    # 320 x 256, the last row of tiles of both problems against the edge, 71 MB
def test_c_of_64_mb_and_more_bit_exact(L, M, N, layout):
    # such a C is read past the caches; D over C
    import torch
    K = 192
    gen = torch.Generator(device="cuda").manual_seed(M + N)
    a, b, c = (torch.randint(-8, 9, shape, generator=gen, device="cuda").half() for shape in ((L, M, K), (L, N, K), (L, M, N)))
    d = c.clone()
    pkg.gemm(a, b if layout == 0 else b.transpose(1, 2).contiguous(), c=d, alpha=0.5, beta=-1.0, layout=layout, out=d)
    torch.cuda.synchronize()
    rows = np.unique(np.concatenate([np.arange(5, M, 173), np.arange(M - 70, M, 3)])).astype(np.int32)
    for i in range(L):
        want = (0.5 * oracle.gemm_f32(*(x[i].float().cpu().numpy() for x in (a, b)), rows=rows) - c[i].float().cpu().numpy()[rows]).astype(np.float16)
        assert np.array_equal(d[i].cpu().numpy()[rows], want), i


@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("L,M,N", [
    (2, 1280, 3328),     # 192 x 192 tiles, the last ones of two problems against both edges
    (1, 1280, 7168),     # 192 x 256, the last row of tiles against the edge
    (1, 2816, 6144)])    # 320 x 256, likewise
def test_macro_tiles_at_an_edge_without_c_bit_exact(L, M, N, layout):
    import torch
    K = 192
    rng = np.random.default_rng(M + N)
    a = rng.integers(-8, 9, (L, M, K)).astype(np.float32)
    b = rng.integers(-8, 9, (L, N, K)).astype(np.float32)
    bt = b if layout == 0 else np.ascontiguousarray(b.transpose(0, 2, 1))
    got = pkg.gemm(to_dev(a.astype(np.float16)), to_dev(bt.astype(np.float16)), layout=layout)
    torch.cuda.synchronize()
    rows = np.unique(np.concatenate([np.arange(3, M, 61), np.arange(M - 70, M)])).astype(np.int32)
    got = got.cpu().numpy()
    for i in range(L):
        assert np.array_equal(got[i][rows], oracle.gemm_f32(a[i], b[i], rows=rows).astype(np.float16)), i


@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("L,M,N", [(1, 4096, 3072), (5, 256, 7168)])   # (the second: the last column of tiles of each problem against the edge)
@pytest.mark.parametrize("K", [1664, 2112])
def test_256_x_192_tiles_bit_exact(L, M, N, K, layout):
    import torch
    gen = torch.Generator(device="cuda").manual_seed(M + N + K)
    a, b, c = (torch.randint(-8, 9, shape, generator=gen, device="cuda").half() for shape in ((L, M, K), (L, N, K), (L, M, N)))
    bt = b if layout == 0 else b.transpose(1, 2).contiguous()
    plain = pkg.gemm(a, bt, layout=layout)
    d = c.clone()
    pkg.gemm(a, bt, c=d, alpha=0.5, beta=-1.0, layout=layout, out=d)
    torch.cuda.synchronize()
    rows = np.arange(3, M, 61).astype(np.int32)
    for i in range(L):
        want = oracle.gemm_f32(*(x[i].float().cpu().numpy() for x in (a, b)), rows=rows)
        assert np.array_equal(plain[i].cpu().numpy()[rows], want.astype(np.float16)), i
        assert np.array_equal(d[i].cpu().numpy()[rows], (0.5 * want - c[i].float().cpu().numpy()[rows]).astype(np.float16)), i


@pytest.mark.parametrize("layout", [0, 1])
def test_an_element_does_not_depend_on_the_tile_it_lies_in(layout):
    # corners of one product over C, each by another macro tile (32 x 32 to 256 x 128, 192 x 192, 192 x 256, 320 x 256; the whole in 256 x 256
    # blocks), with factors that round: one K tile, so that all add up the same products in the same order, and the same bits come out
    import torch
    K = 64
    gen = torch.Generator(device="cuda").manual_seed(12)
    a, b, c = ((torch.rand(shape, generator=gen, device="cuda") * 2 - 1).half() for shape in ((8192, K), (8192, K), (8192, 8192)))
    def product(m, n):
        bt = b[:n] if layout == 0 else b[:n].t().contiguous()
        return pkg.gemm(a[:m], bt, c=c[:m, :n].contiguous(), alpha=1.9, beta=0.707, layout=layout)
    whole = product(8192, 8192)
    for m, n in [(512, 512), (1024, 1024), (1024, 2048), (2048, 2048), (4096, 2048), (3072, 3072), (3072, 4096), (2560, 6656)]:
        assert torch.equal(product(m, n), whole[:m, :n]), (m, n)


def test_fp32_uniform_inputs():
    # the CuTe example's type 1 (float operands, gemm.cu:677-684), U(-1,1) data (:482-485).  Both sides accumulate in
    # fp32 in different orders: |error| <~ sqrt(K) * 2^-24 * |terms|
    import torch
    M, N, K = 512, 256, 4096
    a = pkg.testbed.uniform((M, K), 5).astype(np.float32)
    b = pkg.testbed.uniform((N, K), 6).astype(np.float32)
    want = oracle.gemm_f32(a, b)
    got = pkg.gemm(to_dev(a), to_dev(b))
    torch.cuda.synchronize()
    np.testing.assert_allclose(got.cpu().numpy(), want, rtol=1e-4, atol=2e-4)
    # pins the contraction-slot mapping of the fp32 path against a float64 product on a few rows
    ref64 = a[:8].astype(np.float64) @ b.astype(np.float64).T
    np.testing.assert_allclose(got[:8].cpu().numpy(), ref64, rtol=1e-4, atol=2e-4)


def test_error_paths():
    import torch
    x = torch.zeros((100, 64), dtype=torch.float16, device="cuda:0")
    with pytest.raises(pkg.CfkError) as e:
        pkg.gemm_f16(x, x)
    assert e.value.code == -2
    xf = torch.zeros((256, 64), dtype=torch.float32, device="cuda:0")
    with pytest.raises(pkg.CfkError) as e:      # the N-contiguous B layout is an fp16 layout
        pkg.gemm(xf, torch.zeros((64, 256), dtype=torch.float32, device="cuda:0"), layout=1)
    assert e.value.code == -2
