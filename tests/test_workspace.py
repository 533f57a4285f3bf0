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
        return types.SimpleNamespace(data_ptr=lambda: 0x1000, n=n)


@pytest.mark.parametrize("current", [0, 7])
@pytest.mark.parametrize("stream", [0, 7, 9])
def test_workspace_belongs_to_the_stream_of_the_call(monkeypatch, current, stream):
    fake = FakeTorch(current)
    monkeypatch.setattr(f, "_torch", fake)
    f._workspace(64, stream)
    assert fake.allocated == [(64, stream)] and fake.current == current


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
