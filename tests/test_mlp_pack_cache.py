"""The packed weights that HipMlpLauncher keeps: which change packs them again, and
the order of several streams' and threads' calls around a pack.  On the CPU with a
stand-in for the library and the streams; on the GPU against unpacked weights.
"""

from __future__ import annotations

import ctypes
import threading

import pytest
import torch

from fuseml_amd import _abi
from fuseml_amd.mlp import HipMlpLauncher

BF = torch.bfloat16
M, D, I = 48, 256, 384
gpu = pytest.mark.gpu


class Library(ctypes.CDLL):
    """Counts the packs; its launch meets at `barrier` and then reads the descriptor."""

    def __init__(self, parties=1):
        self.barrier = threading.Barrier(parties)
        self.packs, self.seen = [], {}

    def __getattr__(self, name):  # not ctypes' lookup of a symbol
        raise AttributeError(name)

    def fuseml_mlp_pack_bytes(self, desc_ref):
        return 4 * D * I

    def fuseml_mlp_pack_weights(self, desc_ref, buf, stream):
        self.packs.append((buf.value, stream.value or 0))
        return _abi.OK

    def fuseml_mlp_block(self, desc_ref, stream):
        self.barrier.wait(timeout=20)
        d = ctypes.cast(desc_ref, ctypes.POINTER(_abi.MlpDesc)).contents
        self.seen.setdefault(threading.get_ident(), []).append((d.x, d.w1, d.b1, d.w2, d.y))
        return _abi.OK


class Streams:
    """The streams and events that a pack is ordered by, as a list of what was asked."""

    def __init__(self):
        self.current, self.capturing, self.done, self.log = 1, False, False, []

    def event(self, *args):
        outer = self

        class Event:
            def record(self, stream):
                outer.log.append(("record", stream.cuda_stream))

            def query(self):
                outer.log.append(("query", outer.current))
                return outer.done

        return Event()

    def stream(self, device=None):
        outer = self

        class Stream:
            cuda_stream = outer.current

            def wait_event(self, event):
                outer.log.append(("wait", self.cuda_stream))

        return Stream()


@pytest.fixture
def streams(monkeypatch):
    s = Streams()
    monkeypatch.setattr(torch.cuda, "Event", s.event)
    monkeypatch.setattr(torch.cuda, "current_stream", s.stream)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: s.capturing)
    monkeypatch.setattr(torch.Tensor, "record_stream", lambda t, st: s.log.append(("uses", t.data_ptr(), st.cuda_stream)))
    return s


def _weights():
    return torch.randn(I, D, dtype=BF), torch.randn(D, I, dtype=BF)


def _pack(L, s, w1, w2):
    out = L._packed(None, 4 * D * I, torch.empty(M, D, dtype=BF), w1.t(), w2.t(), s.current)
    return out if isinstance(out, int) else out.data_ptr()


def _launcher(lib):
    L = HipMlpLauncher()
    L._lib = lib
    return L


def test_a_replaced_weight_is_packed(streams):
    """Also where the allocator would give it the freed one's address."""
    L = _launcher(Library())
    for n in range(1, 9):
        w1, w2 = _weights()
        _pack(L, streams, w1, w2)
        assert len(L._lib.packs) == n
        del w1, w2


def test_changes_in_place_and_repack(streams):
    L = _launcher(Library())
    w1, w2 = _weights()
    first = _pack(L, streams, w1, w2)
    assert _pack(L, streams, w1, w2) == first and len(L._lib.packs) == 1
    w2.mul_(2.0)
    _pack(L, streams, w1, w2)
    assert len(L._lib.packs) == 2
    w1.data.mul_(2.0)  # no version shows this one
    L.repack()
    _pack(L, streams, w1, w2)
    assert len(L._lib.packs) == 3


def test_another_stream_waits_for_the_pack_and_keeps_its_buffer(streams):
    L = _launcher(Library())
    w1, w2 = _weights()
    buf = _pack(L, streams, w1, w2)
    assert streams.log == [("record", 1)]
    assert _pack(L, streams, w1, w2) == buf and streams.log == [("record", 1)]
    streams.current = 2
    _pack(L, streams, w1, w2)
    assert streams.log[1:] == [("query", 2), ("wait", 2), ("uses", buf, 2)]
    streams.done = True  # from here on the pack is complete for every stream
    for stream in (3, 2):
        streams.current = stream
        _pack(L, streams, w1, w2)
    assert streams.log[4:] == [("query", 3), ("uses", buf, 3), ("uses", buf, 2)]
    assert len(L._lib.packs) == 1


def test_capture_neither_waits_nor_leaves_its_pack(streams):
    L = _launcher(Library())
    w1, w2 = _weights()
    streams.capturing = True
    _pack(L, streams, w1, w2)         # a node of the graph, filled by its replays
    streams.capturing = False
    _pack(L, streams, w1, w2)
    assert len(L._lib.packs) == 2     # so the first call outside packs for itself
    streams.capturing, streams.current = True, 5
    _pack(L, streams, w1, w2)
    assert len(L._lib.packs) == 2 and streams.log == [("record", 1)]


def test_calls_at_once_have_descriptors_of_their_own(streams, monkeypatch):
    """Host tensors pass for device 0's (nothing dereferences them); a plan's calls
    are held inside the library together."""
    monkeypatch.setattr(torch.Tensor, "get_device", lambda self: 0)
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda index: 1, raising=False)
    n = 4
    L = _launcher(Library(n))
    w1, w2 = _weights()
    b1 = torch.randn(I, dtype=BF)
    xs, got = [torch.randn(M, D, dtype=BF) for _ in range(n)], {}
    # the plan of the signature, as a checked call on a GPU leaves it
    monkeypatch.setattr(HipMlpLauncher, "_launch_checked", lambda *a: pytest.fail("a plan serves every call"))
    key = (xs[0].shape, xs[0].stride(), BF, xs[0].device, w1.t().shape, w1.t().stride(), BF, 0, b1.shape, b1.stride(), BF, 0,
           w2.t().stride(), BF, 0, None, None)
    from fuseml_amd.mlp import _MlpPlan
    L._plans[key] = _MlpPlan(_abi.MlpDesc(), M, D, BF, 4 * D * I)

    def work(i):
        for _ in range(3):
            got.setdefault((i, threading.get_ident()), []).append(L(xs[i], w1.t(), b1, w2.t(), None, None))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(n)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(got) == n
    for (i, ident), outs in got.items():
        assert L._lib.seen[ident] == [(xs[i].data_ptr(), w1.data_ptr(), b1.data_ptr(), w2.data_ptr(), y.data_ptr())
                                      for y in outs]


def _gpu_args(seed, i=I):
    g = torch.Generator().manual_seed(seed)
    t = [torch.randn(M, D, generator=g), torch.randn(i, D, generator=g) / 16, torch.randn(i, generator=g),
         torch.randn(D, i, generator=g) / 16, torch.randn(D, generator=g), torch.randn(M, D, generator=g)]
    x, w1, b1, w2, b2, r = (v.to("cuda", BF) for v in t)
    return x, w1.t(), b1, w2.t(), b2, r


@gpu
def test_replaced_weights_on_the_device():
    L = HipMlpLauncher()
    for seed in range(6):
        args = _gpu_args(seed)  # the weights before these are free memory by now
        assert torch.equal(L(*args), HipMlpLauncher(pack_weights=False)(*args))
        del args


@gpu
def test_weights_that_are_copied_into_place():
    """t(W) laid out row-major is copied per call: the pack follows the weight the
    caller holds, not the copy (whose address comes back every call)."""
    L = HipMlpLauncher()
    x, w1t, b1, w2t, b2, r = _gpu_args(4)
    w1t = w1t.contiguous()
    for _ in range(3):
        args = (x, w1t, b1, w2t, b2, r)
        assert torch.equal(L(*args), HipMlpLauncher(pack_weights=False)(*args))
        pack = L._pack
        L(*args)
        assert L._pack is pack
        w1t.mul_(0.5)


@gpu
def test_streams_around_a_repack():
    """A weight's first call on one stream, the next on others, with changes in
    place between them."""
    L = HipMlpLauncher()
    args = _gpu_args(1, 2048)
    streams = [torch.cuda.Stream() for _ in range(3)]
    outs, wants = [], []
    torch.cuda.synchronize()
    for step in range(12):
        with torch.cuda.stream(streams[step % 3]):
            args[1].mul_(1.03125)
            outs.append(L(*args))
        for other in (1, 2):  # packed just now by another stream
            with torch.cuda.stream(streams[(step + other) % 3]):
                outs.append(L(*args))
        torch.cuda.synchronize()
        wants += [HipMlpLauncher(pack_weights=False)(*args)] * 3
        torch.cuda.synchronize()  # before the weights change again
    for got, want in zip(outs, wants):
        assert torch.equal(got, want)


@gpu
def test_first_call_inside_a_capture():
    args = _gpu_args(3)
    want = HipMlpLauncher(pack_weights=False)(*args)
    HipMlpLauncher()(*args)  # (the kernels are loaded before the capture)
    L = HipMlpLauncher()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = L(*args)
    assert torch.equal(L(*args), want)  # before any replay has filled the graph's own pack
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want) and torch.equal(L(*args), want)
