"""Threads that share a launcher, on the CPU: every call hands the library a
descriptor of its own.  The library is a stand-in whose entry point holds several
calls of one signature inside it at once, as a released interpreter lock may.
"""

from __future__ import annotations

import ctypes
import threading
import warnings

import pytest
import torch

from fuseml_amd import _abi, launcher
from fuseml_amd.epilogue import EpilogueSpec, EpiOp
from fuseml_amd.launcher import _NATIVE_AFTER, HipKernelLauncher

BF = torch.bfloat16
SPEC = EpilogueSpec(1, 2, (EpiOp("add", 0), EpiOp("gelu_erf")), BF)
M, N, K = 16, 24, 32


class Library(ctypes.CDLL):
    """Meets at `barrier` inside the entry point, then reads the descriptor."""

    def __init__(self, parties=1):
        self.barrier = threading.Barrier(parties)
        self.seen = {}

    def __getattr__(self, name):  # not ctypes' lookup of a symbol
        raise AttributeError(name)

    def fuseml_gemm_epilogue(self, desc_ref, stream):
        self.barrier.wait(timeout=20)
        d = ctypes.cast(desc_ref, ctypes.POINTER(_abi.GemmDesc)).contents
        self.seen.setdefault(threading.get_ident(), []).append((d.a, d.lda, d.b, d.operands[0].ptr, d.out.ptr))
        return _abi.OK


class Recorder:
    """The same entry point as a library that is no CDLL: the general path."""

    def __init__(self, parties):
        self.inner = Library(parties)
        self.seen = self.inner.seen

    def fuseml_gemm_epilogue(self, desc_ref, stream):
        return self.inner.fuseml_gemm_epilogue(desc_ref, stream)


class Native:
    """Stands in for the native caller: keeps what is handed over."""

    during = staticmethod(lambda: None)
    plans: list = []

    def __init__(self, *args):
        self.count = 0

    def call(self, inputs):
        return None

    def add(self, inputs, desc, *rest):
        Native.during()
        Native.plans.append(_abi.GemmDesc.from_buffer_copy(desc))
        return True


@pytest.fixture
def on_a_device(monkeypatch):
    """Host tensors pass for device 0 (nothing dereferences them)."""
    monkeypatch.setattr(torch.Tensor, "get_device", lambda self: 0)
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda index: 0, raising=False)
    monkeypatch.setattr(Native, "plans", [])


def _launcher(lib):
    L = HipKernelLauncher(SPEC, 3)
    L._lib = lib
    L._native_type = Native
    return L


def _args(offset=0):
    """Rows of pitch K + 8; `offset` elements into them (3: a base off 16 bytes)."""
    buf = torch.randn(M * (K + 8) + 8, dtype=BF)
    base = -(buf.data_ptr() // 2) % 8 + offset
    x = buf[base:].as_strided((M, K), (K + 8, 1), buf.storage_offset() + base) if base else buf.as_strided((M, K), (K + 8, 1))
    return torch.randn(N, dtype=BF), x, torch.randn(N, K, dtype=BF).t()


@pytest.mark.parametrize("library", [Library, Recorder], ids=["pointers", "general"])
def test_calls_at_once_have_descriptors_of_their_own(library, on_a_device):
    n = 4
    lib = library(n)
    L = _launcher(lib)
    args, got = [_args() for _ in range(n)], {}

    def work(i):
        for _ in range(3):
            got.setdefault((i, threading.get_ident()), []).append(L(*args[i]))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(n)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(got) == n
    for (i, ident), outs in got.items():
        b, x, wt = args[i]
        assert lib.seen[ident] == [(x.data_ptr(), K + 8, wt.data_ptr(), b.data_ptr(), o.data_ptr()) for o in outs]


def test_a_plan_is_handed_over_with_its_own_strides(on_a_device, monkeypatch):
    """While a plan is handed over, another thread's call of its signature may write
    another row stride: a misaligned base is copied to rows of K elements."""
    L = _launcher(Library())
    args, off = _args(), _args(3)
    monkeypatch.setattr(Native, "during", staticmethod(lambda: L.launch(*off)))
    for _ in range(_NATIVE_AFTER + 1):
        L(*args)
    assert off[1].data_ptr() % 16 and off[1].stride() == args[1].stride() and len(L._plans) == 1
    assert [(p.lda, p.ldb) for p in Native.plans] == [(K + 8, K)]


def test_a_plan_is_handed_over_past_its_due_call(on_a_device):
    """Two threads' calls may step past the count at which it is due."""
    L = _launcher(Library())
    args = _args()
    L(*args)
    (plan,) = L._plans.values()
    plan.calls = _NATIVE_AFTER + 5
    for _ in range(3):
        L(*args)
    assert len(Native.plans) == 1


def test_calls_without_the_native_caller(on_a_device, monkeypatch):
    """Where the extension is missing, Python serves every call, with one warning."""
    def missing():
        raise ImportError("no extension")

    monkeypatch.setattr(_abi, "load_fastcall", missing)
    launcher._native_type.cache_clear()
    try:
        with pytest.warns(RuntimeWarning, match="no extension"):
            L = HipKernelLauncher(SPEC, 3)
        with warnings.catch_warnings():
            warnings.simplefilter("error")
            HipKernelLauncher(SPEC, 3)
    finally:
        launcher._native_type.cache_clear()
    L._lib = Library()
    for _ in range(_NATIVE_AFTER + 2):
        L(*_args())
    assert L.launch_count == _NATIVE_AFTER + 2 and L._native is None


def test_entry_addresses_appear_together(monkeypatch):
    """Another thread that asks while they are looked up finds none or both."""
    monkeypatch.setattr(_abi, "_entries", {})
    cast, others = ctypes.cast, []

    def casting(fn, kind):
        if _abi._entries and not others:
            others.append(None)
            others[0] = _abi.entry_address(True)
        return cast(fn, kind)

    monkeypatch.setattr(_abi.ctypes, "cast", casting)
    want = _abi.entry_address(False), _abi.entry_address(True)
    assert all(want) and want[0] != want[1] and set(others) <= {want[1]}
