"""GPU parity of the compiler-scheduled 16x16-MFMA builds (fmha_fwd_kernel16) where the automatic choice takes them: last query
tiles of one to four waves, a few key tiles, and rows whose scores climb over the keys, which sends waves through the slow path of the
row-sum test; of hybrid calls of the same sizes; and of the e4m3 build with pre-transposed V that runs three waves per SIMD.  Gates as in the
other parity tests (max-abs error against fp32 attention, src/fmha-pipeline/fmha_forward.cu:599-683)."""
import math

import numpy as np
import pytest

import oracle
from _util import TOL_FP16, TOL_FP8, climbing_keys, max_abs, pkg, to_dev

pytestmark = pytest.mark.gpu
f = pkg.fmha

# mode, (batch, heads), query rows, head dim, kernel, key lengths
CASES = [
    ("fp16", (2, 8), 5152, 64, "fmha_fwd_kernel16<64,64,4,3,0,", (384, 448, 704)),         # a last tile with one wave
    ("fp16", (2, 8), 5216, 64, "fmha_fwd_kernel16<64,64,4,3,0,", (448,)),                  # ... with three
    ("fp16", (2, 8), 8128, 128, "fmha_fwd_kernel16<128,64,4,2,0,", (384, 576)),            # ... with two
    # hybrid calls of many items run the 32x32 build, whose time does not depend on the scores
    ("hybrid", (1, 8), 16384, 128, "fmha_fwd_kernel<128,64,8,2,1,0,0,0,1,", (64, 128, 192, 1024)),
    ("hybrid", (1, 8), 16384, 128, "fmha_fwd_kernel<128,64,8,2,1,0,0,0,1,", (3072, 3200)),  # an even and an odd number of steps
    ("hybrid", (1, 8), 16384, 64, "fmha_fwd_kernel<64,64,4,3,1,", (1024, 1088)),
    ("e4m3-bdhs", (2, 8), 4256, 64, "fmha_fwd_kernel<64,64,4,3,1,1,1,", (64, 128, 192)),
]


@pytest.mark.parametrize("climb", [False, True])
@pytest.mark.parametrize("mode,bh,Sq,D,kernel,key_lengths", CASES)
def test_partly_filled_tiles_and_few_key_tiles(mode, bh, Sq, D, kernel, key_lengths, climb):
    import torch
    B, H = bh
    for Skv in key_lengths:
        q, k, v = pkg.testbed.qkv(B, Sq, H, D, seqlen_kv=Skv, seed=7)
        if climb:
            k, v = climbing_keys(k, ramp=4.0, spike=4.0), v / 4
        kw, key, tol = {}, dict(dtype=f.CFK_FP8_E4M3), TOL_FP16
        if mode == "fp16":
            key["dtype"] = f.CFK_FP16
            ops = [x.astype(np.float16) for x in (q, k, v)]
            ref = [x.astype(np.float32) for x in ops]
        else:
            codes = [oracle.quantize_e4m3_per_tensor(x) for x in (q, k, v)]
            ref = [oracle.e4m3_decode(c) * s for c, s in codes]
            ops = [c for c, _ in codes]
            kw = dict(q_descale=float(codes[0][1]), k_descale=float(codes[1][1]))
            if mode == "hybrid":
                ops[2], key["v_dtype"] = v.astype(np.float16), f.CFK_FP16
                ref[2] = ops[2].astype(np.float32)
            else:
                kw.update(v_descale=float(codes[2][1]), v_layout=f.CFK_V_BDHS)
                key["v_layout"], tol = f.CFK_V_BDHS, TOL_FP8
                ops[2] = np.ascontiguousarray(ops[2].transpose(0, 3, 2, 1))
        assert f.fmha_forward_kernel(key.pop("dtype"), B, H, Sq, Skv, D, **key).startswith(kernel)
        dev = [to_dev(x) for x in ops]
        o = pkg.fmha_forward(*dev, **kw)
        row_max, row_sum = (torch.zeros((B, H, Sq), dtype=torch.float32, device="cuda:0") for _ in range(2))
        tapped = pkg.fmha_forward(*dev, row_max=row_max, row_sum=row_sum, **kw)
        torch.cuda.synchronize()
        # fp32 attention, one batch entry at a time
        qf, kf, vf = (torch.from_numpy(x).cuda().permute(0, 2, 1, 3).contiguous() for x in ref)
        for b in range(B):
            s = torch.matmul(qf[b], kf[b].transpose(1, 2).contiguous()) / math.sqrt(D)
            want = torch.matmul(torch.softmax(s, -1), vf[b]).permute(1, 0, 2).cpu().numpy()
            for got in (o, tapped):
                err = max_abs(got[b].float().cpu().numpy(), want)
                assert err <= tol, (mode, Sq, Skv, D, climb, b, err)
            # the taps are the row max in the log2 domain and the sum of weights against it: rounded to fp16 or e4m3, whose unbiased
            # roundings move the sum by at most 2^-11 and 2^-4 of it; the score itself is off by up to 2^-14 of its size with e4m3
            # operands (the matrix unit's sum of their products: 5e-5 here, with 32x32 and with 16x16 multiplies alike)
            lse = (row_max[b] + torch.log2(row_sum[b])) * math.log(2.0)
            worst = float((lse - torch.logsumexp(s, -1)).abs().max())
            limit = 2 ** -10 if mode == "fp16" else (2 ** -4 if mode == "e4m3-bdhs" else 2 ** -10) + 2 ** -13 * float(s.abs().max())
            assert worst <= limit, (mode, Sq, Skv, D, climb, b, worst, limit)
