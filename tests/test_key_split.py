"""GPU parity of the key-split kernel (fmha_fwd_kernel_ks: 32 query rows per workgroup, whose waves share the keys) in every
precision mode and head dim, and of the calls whose keys are shared by several workgroups as well (cfk_fmha_forward_ws:
partial results in a workspace, merged by a second kernel).  Key lengths around what the waves' turns divide: fewer tiles
than waves, one each, one more than that, unequal shares.  Oracle and gates as in the other parity tests (max-abs error
against the fp32 host reference attention, src/fmha-pipeline/fmha_forward.cu:599-683)."""
import ctypes

import numpy as np
import pytest

import oracle
from _util import TOL_FP16, TOL_FP8, climbing_keys, max_abs, pkg, to_dev

pytestmark = pytest.mark.gpu
f = pkg.fmha

MODES = ["fp16", "e4m3", "e4m3-bdhs", "hybrid"]


def _operands(mode, B, H, Sq, Skv, D, climb=False, seed=5):
    """(device tensors, keyword arguments, float operands, tolerance, key for the kernel query)"""
    q, k, v = pkg.testbed.qkv(B, Sq, H, D, seqlen_kv=Skv, seed=seed)
    if climb:
        k, v = climbing_keys(k, ramp=4.0, spike=4.0), v / 4
    if mode == "fp16":
        ops = [x.astype(np.float16) for x in (q, k, v)]
        return [to_dev(x) for x in ops], {}, [x.astype(np.float32) for x in ops], TOL_FP16, dict(dtype=f.CFK_FP16)
    (qc, qs), (kc, ks), (vc, vs) = (oracle.quantize_e4m3_per_tensor(x) for x in (q, k, v))
    qf, kf = oracle.e4m3_decode(qc) * qs, oracle.e4m3_decode(kc) * ks
    kw = dict(q_descale=float(qs), k_descale=float(ks))
    if mode == "hybrid":
        v16 = v.astype(np.float16)
        return [to_dev(qc), to_dev(kc), to_dev(v16)], kw, [qf, kf, v16.astype(np.float32)], TOL_FP16, dict(dtype=f.CFK_FP8_E4M3, v_dtype=f.CFK_FP16)
    kw["v_descale"] = float(vs)
    vf = oracle.e4m3_decode(vc) * vs
    if mode == "e4m3-bdhs":
        kw["v_layout"] = f.CFK_V_BDHS
        vc = np.ascontiguousarray(vc.transpose(0, 3, 2, 1))
    return [to_dev(qc), to_dev(kc), to_dev(vc)], kw, [qf, kf, vf], TOL_FP8, dict(dtype=f.CFK_FP8_E4M3, v_layout=kw.get("v_layout", f.CFK_V_BSHD))


def _workspace_bytes(key, B, H, Sq, Skv, D):
    p = f.make_params(key["dtype"], B, H, Sq, Skv, D, v_dtype=key.get("v_dtype"), v_layout=key.get("v_layout", f.CFK_V_BSHD))
    return pkg.lib().cfk_fmha_forward_workspace(ctypes.byref(p))


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("mode", MODES)
def test_key_lengths_around_the_turns_of_the_waves(mode, D):
    import torch
    for Skv in (192, 256, 512, 576, 1088):     # 3 to 17 tiles of 64 keys (up to 34 of 32) for 4 or 8 waves
        B, H, Sq = 2, 3, 96
        dev, kw, ref, tol, key = _operands(mode, B, H, Sq, Skv, D, climb=Skv == 576)
        assert "_ks<" in f.fmha_forward_kernel(key["dtype"], B, H, Sq, Skv, D, v_layout=key.get("v_layout", 0), v_dtype=key.get("v_dtype"))
        row_max, row_sum = (torch.zeros((B, H, Sq), dtype=torch.float32, device="cuda:0") for _ in range(2))
        o = pkg.fmha_forward(*dev, **kw)
        tapped = pkg.fmha_forward(*dev, row_max=row_max, row_sum=row_sum, **kw)
        torch.cuda.synchronize()
        want = oracle.attention_f32(*ref)["O"]
        err = max_abs(o.float().cpu().numpy(), want)
        print(f"{mode} D={D} Skv={Skv}: max-abs {err:.3e}", flush=True)
        assert err <= tol, (mode, D, Skv, err)
        assert max_abs(tapped.float().cpu().numpy(), want) <= tol
        s = np.einsum("bqhd,bkhd->bhqk", ref[0], ref[1]) * (np.log2(np.e) / np.sqrt(D))
        m = s.max(-1)
        # scores up to 50: 1e-4 relative as in the other tap tests, beside the bits that the e4m3 matrix pipe drops when it
        # aligns the products of a step (7.0e-4 at scores of 21, the same figure in every e4m3 build).  The weights are
        # summed in fp32 before their rounding.
        np.testing.assert_allclose(row_max.cpu().numpy(), m, rtol=1e-4, atol=1e-3)
        l = np.exp2(s - m[..., None]).sum(-1)
        np.testing.assert_allclose(row_sum.cpu().numpy(), l, rtol=2e-3)


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("mode", MODES)
def test_keys_shared_by_several_workgroups(mode, D):
    import torch
    for B, H, Sq, Skv, climb in [(1, 1, 32, 8192, False), (2, 2, 96, 4160, True), (1, 3, 160, 6208, False)]:
        dev, kw, ref, tol, key = _operands(mode, B, H, Sq, Skv, D, climb=climb)
        assert _workspace_bytes(key, B, H, Sq, Skv, D) > 0, "the keys of this problem are meant to be split"
        row_max, row_sum = (torch.zeros((B, H, Sq), dtype=torch.float32, device="cuda:0") for _ in range(2))
        o = pkg.fmha_forward(*dev, **kw)
        tapped = pkg.fmha_forward(*dev, row_max=row_max, row_sum=row_sum, **kw)
        torch.cuda.synchronize()
        assert torch.equal(o, tapped)
        s = np.einsum("bqhd,bkhd->bhqk", ref[0], ref[1]) * (np.log2(np.e) / np.sqrt(D))
        np.testing.assert_allclose(row_max.cpu().numpy(), s.max(-1), rtol=1e-4, atol=1e-3)   # (as above)
        np.testing.assert_allclose(row_sum.cpu().numpy(), np.exp2(s - s.max(-1, keepdims=True)).sum(-1), rtol=2e-3)
        err = max_abs(o.float().cpu().numpy(), oracle.attention_f32(*ref)["O"])
        print(f"{mode} D={D} B={B} H={H} Sq={Sq} Skv={Skv}: max-abs {err:.3e}", flush=True)
        assert err <= tol, (mode, D, Skv, err)


def test_workspace_streams_graphs_and_small_workspaces():
    import torch
    B, H, Sq, Skv, D = 1, 2, 64, 4096, 128
    dev, kw, ref, tol, key = _operands("fp16", B, H, Sq, Skv, D)
    want = oracle.attention_f32(*ref)["O"]
    need = _workspace_bytes(key, B, H, Sq, Skv, D)
    assert need > 0
    # a stream of the caller's, as object and as pointer; two streams at once, each call with a workspace of its own
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(2)]
    outs = [pkg.fmha_forward(*dev, stream=st if i % 2 else st.cuda_stream) for i in range(6) for st in streams]
    call = pkg.fmha_forward(*dev, prepare=True)
    for _ in range(3):
        call()
    torch.cuda.synchronize()
    for o in outs + [call.o]:
        assert max_abs(o.float().cpu().numpy(), want) <= tol
    # captured: the workspace is the graph's
    o = torch.zeros_like(outs[0])
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        with torch.cuda.graph(graph, stream=side):
            pkg.fmha_forward(*dev, o=o)
    torch.cuda.current_stream().wait_stream(side)
    for rep in range(3):
        o.fill_(-1.0)
        junk = torch.full((need,), 255, dtype=torch.uint8, device="cuda:0")   # eager work between the replays
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert max_abs(o.float().cpu().numpy(), want) <= tol, rep
        del junk
    # too small a workspace, or none: the call without it; a misaligned one is refused
    p = f.make_params(f.CFK_FP16, B, H, Sq, Skv, D, *(t.data_ptr() for t in dev), o.data_ptr())
    ws = torch.empty(need + 16, dtype=torch.uint8, device="cuda:0")
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for ptr, size in [(None, 0), (ws.data_ptr(), need - 1), (ws.data_ptr(), need)]:
        o.fill_(-1.0)
        assert pkg.lib().cfk_fmha_forward_ws(ctypes.byref(p), ptr, size, stream) == 0
        torch.cuda.synchronize()
        assert max_abs(o.float().cpu().numpy(), want) <= tol
    assert pkg.lib().cfk_fmha_forward_ws(ctypes.byref(p), ws.data_ptr() + 4, need, stream) == -1


@pytest.mark.parametrize("B,H,Sq,Skv,D", [(1, 2, 64, 576, 64), (1, 2, 64, 576, 128), (1, 2, 64, 576, 256), (1, 1, 32, 8192, 128)])
def test_masked_key_ranges(B, H, Sq, Skv, D):
    """Keys taken out by a -inf in K (one element of Q positive throughout): whole tiles of a wave, and of a workgroup where
    the keys are shared, have no finite score.  The first 64 keys stay: every other kernel starts from their row max."""
    import torch
    q, k, v = (x.astype(np.float16) for x in pkg.testbed.qkv(B, Sq, H, D, seqlen_kv=Skv))
    q[..., 0] = 1.0
    k[..., 0] = 0.0
    keep = list(range(64)) + list(range(Skv - 128, Skv - 100))
    masked = np.setdiff1d(np.arange(Skv), keep)
    k[:, masked, :, 0] = -np.inf
    o = pkg.fmha_forward(*(to_dev(x) for x in (q, k, v)))
    torch.cuda.synchronize()
    want = oracle.attention_f32(*(x.astype(np.float32) for x in (q, k[:, keep], v[:, keep])))["O"]
    assert max_abs(o.float().cpu().numpy(), want) <= TOL_FP16


@pytest.mark.parametrize("D,B,H,Sq,Skv", [
    (128, 1, 16, 1024, 8192),   # fewer blocks than CUs: every block cut
    (128, 1, 9, 1312, 8320),    # ... the last one partly filled, key tiles behind the last group of four
    (128, 2, 65, 512, 3328),    # one whole round, 4 further blocks cut
    (64, 2, 8, 1024, 8192),
    (64, 1, 33, 2016, 4160),
    (256, 2, 8, 1024, 4096),
    (256, 1, 37, 928, 2048),
])
@pytest.mark.parametrize("keys", ["plain", "climbing", "masked"])
def test_cut_query_blocks_of_the_hand_scheduled_builds(D, B, H, Sq, Skv, keys):
    import torch
    q, k, v = pkg.testbed.qkv(B, Sq, H, D, seqlen_kv=Skv, seed=7)
    if keys == "climbing":      # weights beyond the fp16 range: the loop that follows the running max
        k, v = climbing_keys(k, ramp=4.0, spike=4.0), v / 4
    q, k, v = (x.astype(np.float16) for x in (q, k, v))
    if keys == "masked":        # whole units without a finite score
        q[..., 0], k[..., 0] = 1.0, 0.0
        k[:, 64:Skv - 96, :, 0] = -np.inf
    dev = [to_dev(x) for x in (q, k, v)]
    assert "16p<" in f.fmha_forward_kernel(f.CFK_FP16, B, H, Sq, Skv, D)
    call = pkg.fmha_forward(*dev, prepare=True)
    assert call._ws_bytes > 0, "query blocks of this problem are meant to be cut"
    o = pkg.fmha_forward(*dev)
    whole = torch.empty_like(o)
    p = f.make_params(f.CFK_FP16, B, H, Sq, Skv, D, *(t.data_ptr() for t in dev), whole.data_ptr())
    assert pkg.lib().cfk_fmha_forward(ctypes.byref(p), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    row_max, row_sum = (torch.zeros((B, H, Sq), dtype=torch.float32, device="cuda:0") for _ in range(2))
    tapped = pkg.fmha_forward(*dev, row_max=row_max, row_sum=row_sum)
    torch.cuda.synchronize()
    # both are within the gate of the exact result
    assert max_abs(o.float().cpu().numpy(), whole.float().cpu().numpy()) <= 2 * TOL_FP16
    for b, h in {(0, 0), (B - 1, H - 1)}:
        qf, kf, vf = (x[b:b + 1, :, h:h + 1].astype(np.float32) for x in (q, k, v))
        if keys == "masked":
            kf, vf = (np.concatenate([x[:, :64], x[:, Skv - 96:]], 1) for x in (kf, vf))
        want = oracle.attention_f32(qf, kf, vf)["O"]
        for got in (o, tapped):
            assert max_abs(got[b:b + 1, :, h:h + 1].float().cpu().numpy(), want) <= TOL_FP16, (b, h)
        s = (qf[0, :, 0] @ kf[0, :, 0].T) * (np.log2(np.e) / np.sqrt(D))
        np.testing.assert_allclose(row_max[b, h].cpu().numpy(), s.max(-1), rtol=1e-4, atol=1e-3)
        np.testing.assert_allclose(row_sum[b, h].cpu().numpy(), np.exp2(s - s.max(-1, keepdims=True)).sum(-1), rtol=2e-3)
