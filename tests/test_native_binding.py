"""The launching calls as native code (csrc/cfk_torch.cpp) against the same calls in Python: the same results for plain calls, and the
same errors for the others, which the native code leaves to Python."""
import contextlib
import os
import subprocess
import types

import pytest
import torch

from _util import ROOT, pkg

f = pkg.fmha


@contextlib.contextmanager
def _in_python(monkeypatch):
    with monkeypatch.context() as m:
        m.setattr(f, "_native", None)
        yield


def test_calls_that_are_not_plain_are_left_to_python():
    f._launchers()
    h, s = torch.zeros((256, 64), dtype=torch.float16), torch.zeros((1, 64, 1, 64), dtype=torch.float16)
    for args in [(h, h, None, 1.0, 0.0, None, 0), (h.to("meta"),) * 2 + (None, 1.0, 0.0, None, 0), (None,) * 7, (1, 2), ()]:
        assert f._native.gemm(*args) is None
    for args in [(s, s, s, None, None, 1.0, 1.0, 1.0, 0, None), (s.to("meta"),) * 3 + (None, None, 1.0, 1.0, 1.0, 0, None), (None,) * 10, ()]:
        assert f._native.fmha(*args) is None


@pytest.mark.parametrize("why", ["missing", "no library", "other torch", "older build"])
def test_calls_go_through_ctypes_where_the_extension_cannot_serve(why, monkeypatch, tmp_path):
    path, version = tmp_path / "cfk_torch.so", str(torch.__version__)
    if why == "no library":
        path.write_bytes(b"not an ELF file")
    if why == "older build":     # (no version in it)
        (tmp_path / "m.c").write_text("#include <Python.h>\nstatic struct PyModuleDef m = {PyModuleDef_HEAD_INIT, \"cfk_torch\", 0, -1, 0};\n"
                                      "PyMODINIT_FUNC PyInit_cfk_torch(void) { return PyModule_Create(&m); }\n")
        subprocess.run(["gcc", "-shared", "-fPIC", "-I", __import__("sysconfig").get_paths()["include"], "-o", str(path), str(tmp_path / "m.c")], check=True)
    if why != "other torch":
        monkeypatch.setattr(f, "_BINDING_PATH", str(path))
    else:
        version = "0.4.1"
    with pytest.warns(RuntimeWarning, match="cfk_torch.so is not used"):
        assert f._load_native(pkg.lib(), version) is None
    monkeypatch.setattr(f, "_native", None)
    h = torch.zeros((256, 64), dtype=torch.float16)
    with pytest.raises(ValueError):    # (the call is made in Python, which refuses a CPU tensor)
        pkg.gemm(h, h)


def _plan(*args):
    r = subprocess.run(["make", "-n", "-B", "-C", os.path.join(ROOT, "cutlass-kernels_amd", "csrc"), *args], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    assert "libcfk_fmha.so" in r.stdout
    return "cfk_torch.so" in r.stdout


def test_the_library_builds_without_torch_or_a_host_compiler():
    assert _plan()
    assert not _plan("PYTHON=false") and not _plan("PYTHON=no-such-python") and not _plan("CXX=no-such-compiler")
    assert not _plan("TORCH=/nowhere") and not _plan("PYINC=/nowhere")


def _gemm_calls():
    gen = torch.Generator("cuda").manual_seed(3)
    m = lambda *shape, dtype=torch.float16: (torch.rand(shape, generator=gen, device="cuda") - 0.5).to(dtype)
    a, b, c = m(256, 192), m(512, 192), m(256, 512)
    yield (a, b), {}
    yield (a, b, c), dict(alpha=2, beta=0.707)
    yield (a, m(192, 512), c), dict(layout=f.CFK_GEMM_NN, beta=1)
    yield (m(3, 256, 64), m(3, 256, 64)), dict(out=m(3, 256, 256))
    yield (m(2, 256, 64, dtype=torch.float32), m(2, 256, 64, dtype=torch.float32), m(2, 256, 256, dtype=torch.float32)), dict(alpha=0.5, beta=-1.0)
    yield (a.requires_grad_(), torch.nn.Parameter(b)), {}
    # errors: of the checks, of the library; what stands for other tensors or other numbers
    yield (a.detach()[:, :64], b[:, :64]), {}
    yield (a, b.float()), {}
    yield (a, b, c[:, :256]), {}
    yield (a, b), dict(layout=7)
    yield (m(200, 64), m(256, 64)), {}
    yield (m(256, 64).t(), m(256, 256)), {}
    yield (m(256, 64, dtype=torch.float32), m(64, 256, dtype=torch.float32)), dict(layout=f.CFK_GEMM_NN)
    yield (a, b, c), dict(alpha=1e300, beta=torch.tensor(1.0))
    yield (a, b), dict(alpha=10**400)
    yield (a, b), dict(alpha="2")


def _fmha_calls():
    gen = torch.Generator("cuda").manual_seed(4)
    r = lambda *shape: torch.randn(shape, generator=gen, device="cuda")
    q, k, v = r(2, 96, 3, 64).half(), r(2, 320, 3, 64).half(), r(2, 320, 3, 64).half()
    q8, k8, v8 = (x.to(torch.float8_e4m3fn) for x in (q, k, v))
    yield (q, k, v), {}
    yield (q, k, v), dict(o=torch.empty_like(q), softmax_scale=1)
    yield (q8, k8, v8), dict(q_descale=0.5, k_descale=2, v_descale=3.0)
    yield tuple(x.view(torch.uint8) for x in (q8, k8, v8)), dict(softmax_scale=0.2)
    yield (q8, k8, v), {}
    yield (q8, k8, v8.view(torch.uint8).permute(0, 3, 2, 1).contiguous().view(torch.float8_e4m3fn)), dict(v_layout=f.CFK_V_BDHS)
    yield (r(1, 32, 2, 128).half(), r(1, 8192, 2, 128).half(), r(1, 8192, 2, 128).half()), {}          # its keys are shared by workgroups
    yield (q.requires_grad_(), k, v), {}
    yield (q.detach()[:, :, :, :32], k, v), {}
    yield (q, k, v8), {}
    yield (q, k, v[:, :64]), {}
    yield (q, k.transpose(1, 2), v), {}
    yield (q, k[:, :300].contiguous(), v[:, :300].contiguous()), {}
    yield (q, k, v), dict(o=torch.empty_like(q, dtype=torch.float32))
    yield (q, k, v), dict(v_layout=f.CFK_V_BDHS)
    yield (q, k, v), dict(softmax_scale=1e300)
    yield (r(1, 64, 1, 0).half(),) * 3, {}


@pytest.mark.gpu
@pytest.mark.parametrize("calls", [_gemm_calls, _fmha_calls])
def test_native_and_python_calls_agree(calls, monkeypatch):
    f._launchers()
    plain, taken = {_gemm_calls: 6, _fmha_calls: 8}[calls], []   # (the first calls of each are plain ones; further ones may reach the library to fail there)
    native_fn = f._native.gemm if calls is _gemm_calls else f._native.fmha

    def noting(*args):
        done = native_fn(*args)
        taken.append(done is not None)
        return done
    monkeypatch.setattr(f, "_native", types.SimpleNamespace(gemm=noting, fmha=noting))
    fn = pkg.gemm if calls is _gemm_calls else pkg.fmha_forward

    def outcome(args, kw):
        try:
            got = fn(*args, **kw)
            assert got is kw.get("out", kw.get("o", got))
            return got.detach().clone(), got.dtype, got.shape, got.stride(), got.requires_grad
        except Exception as e:  # noqa: BLE001
            return type(e), str(e)
    for i, (args, kw) in enumerate(calls()):
        print(f"{fn.__name__} call {i}", flush=True)
        native = outcome(args, kw)
        with _in_python(monkeypatch):
            python = outcome(args, kw)
        torch.cuda.synchronize()
        assert native[1:] == python[1:], i
        if torch.is_tensor(native[0]):
            assert torch.equal(native[0].nan_to_num(), python[0].nan_to_num()), i
        else:
            assert native == python, i
    assert all(taken[:plain]) and len(taken) == i + 1


@pytest.mark.gpu
def test_native_calls_run_on_the_current_stream_and_under_capture():
    a = torch.rand((256, 4096), device="cuda").half()
    f._launchers()
    want = pkg.gemm(a, a)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        late = torch.zeros_like(a)
        torch.cuda._sleep(20_000_000)
        late.copy_(a)
        got = pkg.gemm(late, late)      # (in order behind the copy only on its stream)
    side.synchronize()
    assert torch.equal(got, want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = pkg.gemm(a, a)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
