"""The hand-scheduled fp16 builds with a multiply-add per score (fmha_fwd_kernel16f): every number of key tiles behind the last group of
four, partly filled query tiles, scores that leave the range of fp16 weights, keys shared by several workgroups."""
import json
import os
import subprocess
import sys

import numpy as np
import pytest

import oracle
from _util import ERRPCT_FP16, ROOT, TOL_FP16, climbing_keys, max_abs, pkg, to_dev

f = pkg.fmha

# 8 to 11 tiles: no turn of the loop, then one; 3 x 16 x 2016 rows and 20 x 2016: workgroups that take a second item
WISHES = {
    "256x128/16f": ["f16nt:2,288,2,128,%d" % (64 * t) for t in (8, 9, 10, 11, 13)] + ["f16nt:3,2016,16,128,%d" % k for k in (576, 640, 704)] +
                   ["f16nt:2,288,2,64,%d" % (64 * t) for t in (8, 9, 10, 11, 15)] + ["f16nt:3,2016,16,64,%d" % k for k in (576, 640, 704)] +
                   ["f16ntclimb:2,352,2,%d,%d" % (d, k) for d in (64, 128) for k in (576, 640, 704, 768)] + ["f16ntclimb:5,1024,16,64,640", "f16climb:2,288,2,128,576"],
    "128x128/16f": ["f16nt:2,160,2,%d,%d" % (d, 64 * t) for d in (64, 128) for t in (8, 9, 10, 11)] +
                   ["f16nt:1,2016,20,%d,%d" % (d, k) for d in (64, 128) for k in (576, 640, 704)] + ["f16ntclimb:5,1024,8,128,704", "f16:2,96,2,64,576"],
    "128x64/16f": ["f16nt:2,160,2,256,%d" % (32 * t) for t in (8, 9, 10, 11, 14)] + ["f16nt:3,2016,6,256,%d" % k for k in (288, 320, 352)] +
                  ["f16ntclimb:2,224,2,256,%d" % k for k in (288, 320, 352, 512)] + ["f16:2,96,2,256,320"],
}


@pytest.mark.gpu
@pytest.mark.parametrize("wish", sorted(WISHES))
def test_forced_builds_match_the_oracle(wish):
    env = dict(os.environ, CFK_FMHA_TILE=wish, PYTHONPATH=os.path.join(ROOT, "tests") + os.pathsep + ROOT)
    r = subprocess.run([sys.executable, os.path.join(ROOT, "tests", "tile_case.py"), *WISHES[wish]], env=env, capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stdout + r.stderr
    rows = [json.loads(l.split(" ", 1)[1]) for l in r.stdout.splitlines() if l.startswith("TILECASE ")]
    assert len(rows) == len(WISHES[wish])
    for row in rows:
        assert "%dx%d/16f" % (row["block_m"], row["block_n"]) == wish and row["mfma"] == 16, row
        assert not row["nan"] and row["max_abs"] <= TOL_FP16 and row["err_pct"] <= ERRPCT_FP16, row


def test_which_calls_take_them_without_gpu():
    # where a sum over rounds says less time than for a compiler-scheduled build; not for callers that want a run time independent of the data
    calls = [(7, 23, 192, 6400, 64), (6, 18, 2560, 1856, 128), (2, 8, 8192, 4160, 256), (2, 8, 8192, 8160, 256), (2, 5, 4224, 544, 256), (3, 26, 3328, 1088, 128)]
    for call in calls:
        assert f.fmha_forward_kernel(f.CFK_FP16, *call).startswith("fmha_fwd_kernel16f<"), call
    f.set_option(f.CFK_OPT_PREDICTABLE_LATENCY, 1)
    try:
        for call in calls:
            assert "16f<" not in f.fmha_forward_kernel(f.CFK_FP16, *call) and "16p<" not in f.fmha_forward_kernel(f.CFK_FP16, *call)
            assert pkg.lib().cfk_fmha_forward_workspace(f.make_params(f.CFK_FP16, *call)) == 0
    finally:
        f.set_option(f.CFK_OPT_PREDICTABLE_LATENCY, 0)
    for call in [(5, 16, 1696, 3584, 64), (8, 16, 2048, 2048, 128), (2, 8, 8192, 8192, 256)]:   # whole groups of four tiles: the scale in Q
        assert f.fmha_forward_kernel(f.CFK_FP16, *call).startswith("fmha_fwd_kernel16p<"), call


# where the sums over rounds say less time for these builds and the calls took more: 1.02 to 1.37 of the compiler-scheduled builds' (fmha_fwd_f16.hip)
SLOWER = [(5, 60, 128, 1152, 64), (8, 43, 128, 1472, 64), (6, 37, 128, 1216, 64), (7, 24, 96, 1088, 64), (8, 30, 160, 640, 64), (3, 54, 256, 576, 64),
          (4, 24, 608, 1728, 128), (8, 18, 576, 1216, 128), (3, 48, 288, 3520, 128), (3, 20, 288, 1152, 128), (7, 48, 224, 768, 128), (8, 4, 2912, 704, 128)]
FASTER = [(3, 27, 224, 1408, 64), (8, 10, 192, 1856, 64), (7, 29, 160, 1024, 64), (5, 27, 160, 832, 64), (6, 17, 160, 1728, 128), (3, 32, 192, 1856, 128),
          (2, 22, 2208, 640, 128), (5, 38, 192, 2112, 128), (8, 20, 160, 2944, 128)]   # 0.82 to 0.96, on the other side of the lines


def test_calls_that_these_builds_lose_stay_compiler_scheduled_without_gpu():
    for call in SLOWER:
        assert f.fmha_forward_kernel(f.CFK_FP16, *call).startswith(("fmha_fwd_kernel<", "fmha_fwd_kernel16<")), call
    for call in FASTER:
        assert f.fmha_forward_kernel(f.CFK_FP16, *call).startswith("fmha_fwd_kernel16f<"), call


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,Sq,Skv,D", [(2, 18, 2016, 3200, 128), (1, 50, 192, 1984, 128), (1, 18, 3840, 3264, 64), (1, 4, 1504, 4672, 256), (1, 4, 1216, 1696, 256)])
@pytest.mark.parametrize("keys", ["plain", "climbing", "masked"])
def test_cut_calls(B, H, Sq, Skv, D, keys):
    import torch
    q, k, v = pkg.testbed.qkv(B, Sq, H, D, seqlen_kv=Skv, seed=11)
    if keys == "climbing":
        k, v = climbing_keys(k, ramp=4.0, spike=4.0), v / 4
    q, k, v = (x.astype(np.float16) for x in (q, k, v))
    if keys == "masked":        # whole units without a finite score
        q[..., 0], k[..., 0] = 1.0, 0.0
        k[:, 64:Skv - 96, :, 0] = -np.inf
    dev = [to_dev(x) for x in (q, k, v)]
    assert "16p<" not in f.fmha_forward_kernel(f.CFK_FP16, B, H, Sq, Skv, D)
    call = pkg.fmha_forward(*dev, prepare=True)
    assert call._ws_bytes > 0, "query blocks of this problem are meant to be cut"
    o = call()
    torch.cuda.synchronize()
    for b, h in {(0, 0), (B - 1, H - 1)}:
        qf, kf, vf = (x[b:b + 1, :, h:h + 1].astype(np.float32) for x in (q, k, v))
        if keys == "masked":
            kf, vf = (np.concatenate([x[:, :64], x[:, Skv - 96:]], 1) for x in (kf, vf))
        want = oracle.attention_f32(qf, kf, vf)["O"]
        got = o[b:b + 1, :, h:h + 1].float().cpu().numpy()
        assert max_abs(got, want) <= TOL_FP16, (b, h)
        if keys == "plain":     # no second rounding of Q: weights and output as rounded to fp16, 2.9e-4 of the size of O (with it 3.6e-4)
            assert np.linalg.norm(got - want) <= 3.2e-4 * np.linalg.norm(want)
