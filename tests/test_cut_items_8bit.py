"""Calls with e4m3 Q and K some of whose items are cut along the keys (SplitCfg builds of fmha_fwd_kernel: partial results in a
workspace, merged by a second kernel): every build that is cut, items cut all and behind whole ones, shares of unequal length, a last
tile of query rows that is partly filled.  Oracle and gates as in the other parity tests (max-abs error and error percentage against the
fp32 host reference attention, src/fmha-pipeline/fmha_forward.cu:599-683)."""
import ctypes

import numpy as np
import pytest

import oracle
from _util import ERRPCT_FP16, ERRPCT_FP8, TOL_FP16, TOL_FP8, climbing_keys, max_abs, pkg, to_dev

f = pkg.fmha

CALLS = [  # mode, D, heads, rows, keys, query blocks that stay whole
    ("e4m3", 64, 8, 3168, 6656, 0), ("e4m3", 64, 34, 2848, 3840, 768), ("e4m3-bdhs", 64, 8, 3168, 6336, 0), ("e4m3-bdhs", 64, 34, 2880, 3584, 768),
    ("e4m3-bdhs", 64, 18, 1024, 6080, 0), ("e4m3-bdhs", 64, 9, 2208, 4992, 0),   # (up to 512 units: the build with two waves per SIMD)
    ("e4m3", 128, 4, 2144, 3136, 0), ("e4m3", 128, 23, 2880, 3072, 512), ("e4m3-bdhs", 128, 4, 2272, 3136, 0), ("e4m3-bdhs", 128, 22, 3008, 3136, 512),
    ("e4m3", 256, 4, 2080, 1152, 0), ("e4m3", 256, 4, 2112, 1280, 0), ("e4m3", 256, 12, 3104, 1088, 256),
    ("e4m3-bdhs", 256, 4, 2240, 1344, 0), ("e4m3-bdhs", 256, 14, 2592, 1216, 256), ("e4m3-bdhs", 256, 4, 2272, 3136, 0),
    ("hybrid", 64, 7, 2464, 5120, 0), ("hybrid", 64, 33, 2976, 2944, 768), ("hybrid", 128, 4, 2208, 1984, 0), ("hybrid", 128, 22, 3104, 2752, 512),
    ("hybrid", 256, 4, 2080, 1408, 0), ("hybrid", 256, 12, 2848, 1344, 256),
]


def _params(mode, D, H, Sq, Skv, *pointers, **kw):
    return f.make_params(f.CFK_FP8_E4M3, 1, H, Sq, Skv, D, *pointers, v_dtype=f.CFK_FP16 if mode == "hybrid" else None,
                         v_layout=f.CFK_V_BDHS if mode == "e4m3-bdhs" else f.CFK_V_BSHD, **kw)


@pytest.mark.parametrize("mode,D,H,Sq,Skv,whole", CALLS)
def test_how_calls_are_cut(mode, D, H, Sq, Skv, whole):
    workspace = lambda **kw: pkg.lib().cfk_fmha_forward_workspace(ctypes.byref(_params(mode, D, H, Sq, Skv, **kw)))
    blocks = H * -(-Sq // 128)
    n, rest = divmod(workspace(), (blocks - whole) * 128 * (D + 2) * 4)
    assert rest == 0 and n >= 2
    assert n * (blocks - whole) <= {64: 3, 128: 2, 256: 1}[D] * 256   # (all on the chip at once)
    assert workspace(dbg_row_max=1) == workspace(dbg_row_sum=1) == workspace(dbg_s=1) == 0   # (the taps are against the row max)
    if mode == "e4m3-bdhs" and D == 64:   # (which of two builds runs the units)
        assert (whole + n * (blocks - whole) <= 512) == ((H, Sq) in {(18, 1024), (9, 2208)})
    if mode != "hybrid":   # (another first pass)
        try:
            f.set_option(f.CFK_OPT_FAST_E4M3_WEIGHTS, 1)
            assert workspace() == 0
        finally:
            f.set_option(f.CFK_OPT_FAST_E4M3_WEIGHTS, 0)


def test_calls_of_the_key_split_kernel_stay_there():
    # (its weights have 16 bits)
    for mode, D in (("e4m3", 64), ("e4m3-bdhs", 128), ("e4m3", 256), ("hybrid", 256)):
        p = _params(mode, D, 20, 160, 7872)
        assert "_ks<" in f.fmha_forward_kernel(p.dtype, 1, 20, 160, 7872, D, v_layout=p.v_layout, v_dtype=p.v_dtype)
        assert pkg.lib().cfk_fmha_forward_workspace(ctypes.byref(p)) % (20 * 160 * (D + 2) * 4) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("mode,D,H,Sq,Skv,whole", CALLS)
@pytest.mark.parametrize("keys", ["plain", "climbing"])
def test_cut_calls(mode, D, H, Sq, Skv, whole, keys):
    import torch
    q, k, v = pkg.testbed.qkv(1, Sq, H, D, seqlen_kv=Skv, seed=11)
    if keys == "climbing":      # weights beyond the range of the first pass: units that walk their keys again
        k, v = climbing_keys(k, ramp=4.0, spike=4.0), v / 4
    (qc, qs), (kc, ks) = (oracle.quantize_e4m3_per_tensor(x) for x in (q, k))
    kw, tol = dict(q_descale=float(qs), k_descale=float(ks)), TOL_FP16
    if mode == "hybrid":
        v_dev, vf = v.astype(np.float16), v.astype(np.float16).astype(np.float32)
    else:
        vc, vs = oracle.quantize_e4m3_per_tensor(v)
        kw["v_descale"], tol, vf = float(vs), TOL_FP8, oracle.e4m3_decode(vc) * vs
        if mode == "e4m3-bdhs": kw["v_layout"] = f.CFK_V_BDHS
        v_dev = np.ascontiguousarray(vc.transpose(0, 3, 2, 1)) if mode == "e4m3-bdhs" else vc
    dev = [to_dev(x) for x in (qc, kc, v_dev)]
    call = pkg.fmha_forward(*dev, prepare=True, **kw)
    assert call._ws_bytes > 0, "query blocks of this problem are meant to be cut"
    o = pkg.fmha_forward(*dev, **kw)
    uncut = torch.empty_like(o)
    p = _params(mode, D, H, Sq, Skv, *(t.data_ptr() for t in dev), uncut.data_ptr(), **{x: kw[x] for x in kw if x != "v_layout"})
    assert pkg.lib().cfk_fmha_forward(ctypes.byref(p), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    call()
    torch.cuda.synchronize()
    assert torch.equal(call.o, o)
    assert max_abs(o.float().cpu().numpy(), uncut.float().cpu().numpy()) <= 2 * tol   # both are within the gate of the exact result
    pct = {"cut": 0.0, "uncut": 0.0}
    for h in (0, H - 1):
        qf, kf = oracle.e4m3_decode(qc[:, :, h:h + 1]) * qs, oracle.e4m3_decode(kc[:, :, h:h + 1]) * ks
        want = oracle.attention_f32(qf, kf, vf[:, :, h:h + 1])["O"]
        err = max_abs(o[:, :, h:h + 1].float().cpu().numpy(), want)
        for name, t in (("cut", o), ("uncut", uncut)): pct[name] += oracle.verify_tensor(t[:, :, h:h + 1].float().cpu().numpy(), want)[1] / 2
        print(f"{mode} D={D} {H} x {Sq} x {Skv} head {h} {keys}: max-abs {err:.3e}", flush=True)
        assert err <= tol
    print(f"    error % cut {pct['cut']:.2e}, uncut {pct['uncut']:.2e}", flush=True)
    # The reference's own gate.  With e4m3 weights it is calibrated for its 4096 keys of N(0,1) scores, and held from 3072 on, where the pass
    # starts whose reference point is the first tile's -- of a unit now, of three tiles or more; over fewer keys, and where a handful
    # of keys carry a row, the rounding of a few weights shows in every such kernel: cut no more of it than uncut.
    if mode == "hybrid":
        assert pct["cut"] <= ERRPCT_FP16
    elif keys == "plain" and Skv >= 3072:
        assert pct["cut"] <= ERRPCT_FP8
    else:
        assert pct["cut"] <= pct["uncut"] + ERRPCT_FP8
