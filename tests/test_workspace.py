"""Where the scratch memory of a call comes from (cfk_fmha_forward_ws through the Python binding): torch's allocator, for the stream
that the call runs on and for as long as the call, or a graph that holds it, can run.  Without a GPU torch is played by a stand-in
that notes what is asked of it."""
import contextlib
import types

import numpy as np
import pytest

import oracle
from _util import TOL_FP16, max_abs, pkg, to_dev

f = pkg.fmha
SPLIT = (1, 2, 64, 4096, 128)      # batch, heads, query rows, keys, head dim: the keys of this fp16 call are split


class FakeTorch:
    """torch as ``_workspace`` sees it: streams are their pointers; ``allocated`` holds (bytes, stream at the allocation)."""
    uint8 = "uint8"

    class OutOfMemoryError(RuntimeError):
        pass

    def __init__(self, current=0):
        self.current, self.allocated = current, []
        self._C = types.SimpleNamespace(_cuda_getDevice=lambda: 0, _cuda_getCurrentRawStream=lambda dev: self.current)
        # (as torch does: a zero pointer is "none given" to ExternalStream, which answers with a stream of its pool)
        self.cuda = types.SimpleNamespace(stream=self._stream, default_stream=lambda dev: 0, ExternalStream=lambda p, device: p or 0xb001)

    def device(self, kind, index):
        return f"{kind}:{index}"

    @contextlib.contextmanager
    def _stream(self, s):
        before, self.current = self.current, s
        yield
        self.current = before

    def empty(self, n, dtype, device):
        self.allocated.append((n, self.current))
        address = 0x1000 * len(self.allocated)
        return types.SimpleNamespace(data_ptr=lambda: address, n=n)


@pytest.mark.parametrize("current", [0, 7])
@pytest.mark.parametrize("stream", [0, 7, 9])
def test_workspace_belongs_to_the_stream_of_the_call(monkeypatch, current, stream):
    fake = FakeTorch(current)
    monkeypatch.setattr(f, "_torch", fake)
    f._workspace(64, stream)
    assert fake.allocated == [(64, stream)] and fake.current == current


def _prepared(monkeypatch, fake, stream):
    """A prepared split call of the real library's plan on a stand-in torch, and the (workspace, bytes) of its launches."""
    launches = []
    monkeypatch.setattr(f, "_torch", fake)
    B, H, Sq, Skv, D = SPLIT
    call = f.PreparedForward(f.make_params(f.CFK_FP16, B, H, Sq, Skv, D), (None,) * 7, stream)
    call._fn = lambda ref, ws, n, stream: launches.append((ws, n)) or 0
    return call, launches


def test_captured_prepared_call_has_scratch_memory_of_the_graph(monkeypatch):
    # (what the object keeps dies with it, while the graph can still be replayed)
    fake, capturing = FakeTorch(), []
    monkeypatch.setattr(f, "_is_capturing", lambda stream: bool(capturing), raising=False)
    call, launches = _prepared(monkeypatch, fake, 7)
    call()
    kept = list(fake.allocated)
    capturing.append(True)
    call(), call()
    capturing.clear()
    call()
    need = kept[0][0]
    assert kept == [(need, 7)] and fake.allocated == [(need, 7)] * 3
    addresses = [ws for ws, _ in launches]
    assert addresses[0] == addresses[3] and len(set(addresses)) == 3 and all(n == need for _, n in launches)


@pytest.mark.parametrize("capturing", [False, True])
def test_prepared_call_without_room_for_scratch_memory_runs_without_it(monkeypatch, capturing):
    fake = FakeTorch()

    def empty(*args, **kw):
        raise FakeTorch.OutOfMemoryError
    fake.empty = empty
    monkeypatch.setattr(f, "_is_capturing", lambda stream: capturing)
    call, launches = _prepared(monkeypatch, fake, 7)
    call()
    assert [ws for ws, _ in launches] == [None]


class _NotingTorch:
    """torch, noting on which stream ``empty`` is called for bytes."""

    def __init__(self, torch):
        self._torch, self.streams = torch, []

    def __getattr__(self, name):
        return getattr(self._torch, name)

    def empty(self, *args, **kw):
        if kw.get("dtype") is self._torch.uint8:
            self.streams.append(self._torch.cuda.current_stream().cuda_stream)
        return self._torch.empty(*args, **kw)


def _operands():
    B, H, Sq, Skv, D = SPLIT
    ops = [x.astype(np.float16) for x in pkg.testbed.qkv(B, Sq, H, D, seqlen_kv=Skv, seed=5)]
    return [to_dev(x) for x in ops], oracle.attention_f32(*(x.astype(np.float32) for x in ops))["O"]


@pytest.mark.gpu
def test_workspace_belongs_to_the_stream_of_the_call_gpu(monkeypatch):
    import torch
    dev, want = _operands()
    f._launchers()
    noting = _NotingTorch(torch)
    monkeypatch.setattr(f, "_torch", noting)
    torch.cuda.synchronize()
    side, other = torch.cuda.Stream(), torch.cuda.Stream()
    outs, streams = [], [0, side.cuda_stream, other, other.cuda_stream, None]
    with torch.cuda.stream(side):
        for s in streams:
            outs.append(pkg.fmha_forward(*dev, stream=s))
            call = pkg.fmha_forward(*dev, stream=s, prepare=True)
            outs.append(call())
    torch.cuda.synchronize()
    expect = [0, side.cuda_stream, other.cuda_stream, other.cuda_stream, side.cuda_stream]
    assert noting.streams == [s for s in expect for _ in range(2)]
    for o in outs:
        assert max_abs(o.float().cpu().numpy(), want) <= TOL_FP16


@pytest.mark.gpu
def test_graph_outlives_the_prepared_call_that_it_captured():
    import torch
    dev, want = _operands()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    o = torch.zeros_like(dev[0])
    call = pkg.fmha_forward(*dev, o=o, stream=side, prepare=True)
    need = call._ws_bytes
    assert need > 0
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        assert f._is_capturing(call._stream)
        call()
    assert not f._is_capturing(call._stream)
    torch.cuda.synchronize()
    del call
    for rep in range(3):
        with torch.cuda.stream(side):      # what the object kept is free: other tensors of its stream
            others = [torch.full((need,), 77, dtype=torch.uint8, device="cuda:0") for _ in range(4)]
        o.fill_(-1.0)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert max_abs(o.float().cpu().numpy(), want) <= TOL_FP16, rep
        assert all(bool((x == 77).all()) for x in others), rep
