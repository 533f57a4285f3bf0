"""fmha_combine over every number of parts that it has code of its own for, and more: fp16 calls whose keys are cut into that many units of
work, by the key-split kernel (32 rows) and by the hand-scheduled ones (128 and 256), against the fp32 oracle."""
import ctypes

import numpy as np
import pytest

import oracle
from _util import TOL_FP16, max_abs, pkg, to_dev

# parts, rows of a unit, heads, query rows, keys, head dim
CUT = [(2, 128, 8, 384, 3072, 128), (2, 128, 8, 384, 1024, 256), (3, 256, 4, 384, 2048, 128), (3, 32, 6, 256, 768, 256), (4, 32, 1, 32, 4096, 64),
       (4, 128, 4, 384, 4096, 64), (5, 128, 4, 384, 3072, 256), (6, 32, 1, 32, 768, 256), (6, 128, 18, 512, 3072, 64),
       (7, 32, 1, 32, 3584, 128), (7, 128, 2, 64, 3584, 256), (7, 128, 2, 256, 3584, 64), (8, 32, 1, 32, 4096, 128),
       (11, 32, 1, 32, 8192, 128), (16, 32, 1, 32, 4096, 256)]


def _parts(bm, H, Sq, Skv, D):
    p = pkg.fmha.make_params(pkg.fmha.CFK_FP16, 1, H, Sq, Skv, D)
    return pkg.lib().cfk_fmha_forward_workspace(ctypes.byref(p)) / (H * -(-Sq // bm) * bm * (D + 2) * 4)


def test_every_number_of_parts_with_code_of_its_own_is_in_the_list():
    assert {n for n, *_ in CUT} > set(range(2, 9)) and max(CUT)[0] > 8


@pytest.mark.parametrize("n,bm,H,Sq,Skv,D", CUT)
def test_calls_are_cut_into_so_many_parts(n, bm, H, Sq, Skv, D):
    assert _parts(bm, H, Sq, Skv, D) == n


@pytest.mark.gpu
@pytest.mark.parametrize("n,bm,H,Sq,Skv,D", CUT)
def test_merge_of_parts(n, bm, H, Sq, Skv, D):
    rng = np.random.default_rng(n * 1000 + D)
    q, k, v = (rng.standard_normal((1, s, H, D)).astype(np.float16) for s in (Sq, Skv, Skv))
    k[:, :Skv // n] *= np.float16(1.5)   # (the parts' reference points and sums are apart)
    want = oracle.attention_f32(*(x.astype(np.float32) for x in (q, k, v)))["O"]
    o = pkg.fmha_forward(*(to_dev(x) for x in (q, k, v)))
    assert max_abs(o.float().cpu().numpy(), want) <= TOL_FP16
