"""The launchers' native calls (csrc/fastcall.cpp): which calls they serve, and
that what they serve is what the Python path gives.  The GPU tests compare the
two on the device; the rest needs none.
"""

from __future__ import annotations

import struct
import threading

import pytest
import torch

from fuseml_amd import _abi
from fuseml_amd.epilogue import EpilogueSpec, EpiOp
from fuseml_amd.fallback import FORCE_FAIL_ENV
from fuseml_amd.launcher import _NATIVE_AFTER, HipKernelLauncher

BF = torch.bfloat16
SPEC = EpilogueSpec(1, 2, (EpiOp("add", 0), EpiOp("gelu_erf")), BF)


def _args(M=32, N=264, K=128, device="cpu", dtype=BF):
    g = torch.Generator().manual_seed(M * 7 + N)
    b, x, w = torch.randn(N, generator=g), torch.randn(M, K, generator=g), torch.randn(N, K, generator=g) / K ** 0.5
    return b.to(device, dtype), x.to(device, dtype), w.to(device, dtype).t()


def test_host_tensors_and_unknown_calls_are_declined():
    fast = _abi.load_fastcall()(3, (0, 1, 2), False)
    args = _args()
    assert fast.call(args) is None and fast.call(args[:2]) is None and fast.call([*args]) is None
    desc = bytes(_abi.GemmDesc())
    # a plan for host tensors is not taken
    assert fast.add(args, desc, 1, 1, 2, ((0, 0),), BF, (), (), (("t", 0),)) is False
    assert fast.call(args) is None and fast.count == 0


@pytest.mark.parametrize("bad", [
    dict(desc=b"short"), dict(left=3), dict(right=-1), dict(operands=((9, 0),)), dict(operands=((0, 5),)),
    dict(reductions=(3,)), dict(reductions=(0, 1, 2, 0)), dict(outputs=()), dict(outputs=(("r", 0),)),
    dict(outputs=(("x", 0),)), dict(extras=(BF,) * 5)])
def test_malformed_plans_are_refused(bad):
    """No plan reaches the list whose call could write outside its descriptor
    (with tensors a plan is not taken for, so a wrong acceptance shows as False)."""
    fast = _abi.load_fastcall()(3, (0, 1, 2), False)
    a = dict(desc=bytes(_abi.GemmDesc()), left=1, right=2, operands=((0, 0),), extras=(), reductions=(),
             outputs=(("t", 0),)) | bad
    checked_late = {"operands", "outputs"} & set(bad) or bad.get("reductions") == (3,)
    try:
        taken = fast.add(_args(), a["desc"], 1, a["left"], a["right"], a["operands"], BF, a["extras"],
                         a["reductions"], a["outputs"])
    except ValueError:
        return
    assert checked_late and taken is False


def test_the_extension_has_no_thread_local_storage():
    """Its ELF program headers hold no PT_TLS (7): see build.fastcall_command."""
    from fuseml_amd.build import FASTCALL_PATH

    with open(FASTCALL_PATH, "rb") as f:
        head = f.read(64)
        offset, = struct.unpack_from("<Q", head, 32)
        size, count = struct.unpack_from("<HH", head, 54)
        f.seek(offset)
        table = f.read(size * count)
    assert head[:5] == b"\x7fELF\x02"
    assert 7 not in [struct.unpack_from("<I", table, size * i)[0] for i in range(count)]


gpu = pytest.mark.gpu


def _python(launcher, args):
    return launcher.launch(*args)


@gpu
@pytest.mark.parametrize("dtype", [BF, torch.float16, torch.float32], ids=["bf16", "fp16", "fp32"])
def test_native_call_is_the_python_call(dtype):
    spec = EpilogueSpec(1, 2, (EpiOp("add", 0), EpiOp("store", 0), EpiOp("relu")), dtype, extra_dtypes=(torch.float32,),
                        reductions=("sum", "amax"), reduce_axis=1, reduce_dtypes=(torch.float32,) * 2,
                        outputs=(("red", "amax"), ("tile",), ("extra", 0), ("red", "sum")))
    L = HipKernelLauncher(spec, 3)
    for M, N in ((32, 264), (300, 520), (32, 264), (1, 8)):
        args = _args(M, N, device="cuda", dtype=dtype)
        first = L(*args)
        for _ in range(_NATIVE_AFTER - 1):
            L(*args)                 # then the signature's plan is handed over
        before = L._native.count
        got = L(*args)
        assert L._native.count == before + 1
        want = _python(L, args)
        for f, g, w in zip(first, got, want):
            assert g.shape == w.shape and g.dtype == w.dtype and g.is_contiguous()
            torch.testing.assert_close(g, w, rtol=1e-6, atol=1e-6)  # fp32 sums by atomics
            torch.testing.assert_close(f, w, rtol=1e-6, atol=1e-6)
        assert got[1].data_ptr() != first[1].data_ptr()
    assert L.launch_count == 4 * (_NATIVE_AFTER + 2)


@gpu
def test_declined_forms_give_the_same_result():
    """Misaligned bases, layouts that need a copy, parameters, subclasses, inputs
    on other devices, a forced failure and the timing hook."""
    L = HipKernelLauncher(SPEC, 3, eager_fn=lambda b, x, w: torch.nn.functional.gelu(torch.addmm(b, x, w)))
    b, x, wt = _args(device="cuda")
    want = L(b, x, wt)
    for _ in range(_NATIVE_AFTER):
        L(b, x, wt)
    n = L._native.count
    assert n == 1
    off = torch.empty(x.shape[0], x.shape[1] + 8, dtype=BF, device="cuda")[:, 3:-5].copy_(x)
    assert torch.equal(L(b, off, wt), want)
    # a misaligned contiguous operand has no kernel: the eager path, as ever
    off = torch.empty(x.numel() + 1, dtype=BF, device="cuda")[1:].view_as(x).copy_(x)
    torch.testing.assert_close(L(b, off, wt).float(), want.float(), rtol=2e-2, atol=2e-2)
    assert L.fallback_count == 1
    assert torch.equal(L(b, x, wt.contiguous()), want)

    class Sub(torch.Tensor):
        pass

    assert torch.equal(L(b, x.as_subclass(Sub), wt).as_subclass(torch.Tensor), want)
    assert L._native.count == n
    p = torch.nn.Parameter(wt.t(), requires_grad=False)
    assert torch.equal(L(b, x, p.t()), want) and torch.equal(L(torch.nn.Parameter(b), x, wt), want)
    assert L._native.count == n + 2
    L.timing_events = []
    assert torch.equal(L(b, x, wt), want) and len(L.timing_events) == 1 and L._native.count == n + 2
    L.timing_events = None
    with pytest.raises(ValueError):
        L(b, x)
    fb = L.fallback_count
    with pytest.MonkeyPatch.context() as mp:
        mp.setenv(FORCE_FAIL_ENV, "1")
        torch.testing.assert_close(L(b, x, wt).float(), want.float(), rtol=2e-2, atol=2e-2)
    assert L.fallback_count == fb + 1
    with pytest.raises(RuntimeError):
        HipKernelLauncher(SPEC, 3)(b.cpu(), x, wt)
    batched = torch.stack([x, x])
    with pytest.raises(RuntimeError):  # no batching rule: refused, as the Python path refuses it
        torch.vmap(lambda v: HipKernelLauncher(SPEC, 3)(b, v, wt))(batched)


@gpu
def test_more_signatures_than_native_plans():
    L = HipKernelLauncher(SPEC, 3)
    b, x, wt = _args(M=200, device="cuda")
    full = L(b, x, wt)
    for m in range(1, 100):
        for _ in range(_NATIVE_AFTER + 1):
            torch.testing.assert_close(L(b, x[:m], wt).float(), full[:m].float(), rtol=2 ** -7, atol=2 ** -7)
    assert L.launch_count == 1 + (_NATIVE_AFTER + 1) * 99 and L._native.count == 64


@gpu
def test_threads_and_streams_share_a_launcher():
    """Four threads, each on a stream of its own with inputs of its own, through
    one launcher and one signature: each gets its own result."""
    L = HipKernelLauncher(SPEC, 3)
    ins = []
    for t in range(4):
        b, x, wt = _args(M=64, device="cuda")
        ins.append((b, x * (t + 1), wt))
    want = [L(*a) for a in ins]
    torch.cuda.synchronize()
    bad = []

    def work(t):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(200):
                if not torch.equal(L(*ins[t]), want[t]):
                    bad.append(t)
                    return

    threads = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


@gpu
def test_threads_share_a_launcher_from_its_first_call():
    """The same without a call made before: calls of the Python path, the plan's
    handover and native calls run at once, two threads' rows off 16 bytes (copied
    per call) under the others' signature."""
    M, N, K = 64, 264, 128
    b, _, wt = _args(M, N, K, device="cuda")
    ins, want = [], []
    for t in range(4):
        rows = torch.zeros(M * (K + 8) + 8, dtype=BF, device="cuda")[3 * (t % 2):].as_strided((M, K), (K + 8, 1))
        rows.copy_(torch.randn(M, K, generator=torch.Generator().manual_seed(t)).to(BF))
        ins.append((b, rows, wt))
        want.append(HipKernelLauncher(SPEC, 3)(b, rows.contiguous(), wt))
    torch.cuda.synchronize()
    for _ in range(20):
        L, bad = HipKernelLauncher(SPEC, 3), []
        start = threading.Barrier(4)

        def work(t):
            with torch.cuda.stream(torch.cuda.Stream()):
                start.wait()
                outs = [L(*ins[t]) for _ in range(12)]
                torch.cuda.current_stream().synchronize()
                bad.extend(t for o in outs if not torch.equal(o, want[t]))

        threads = [threading.Thread(target=work, args=(t,)) for t in range(4)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not bad and len(L._plans) == 1


@gpu
def test_native_call_in_a_graph_replays():
    L = HipKernelLauncher(SPEC, 3)
    b, x, wt = _args(device="cuda")
    for _ in range(_NATIVE_AFTER + 1):
        L(b, x, wt)
    assert L._native.count == 1
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = L(b, x, wt)
    for seed in range(3):
        x.copy_(torch.randn(x.shape, generator=torch.Generator().manual_seed(seed)).to(BF))
        want = L(b, x, wt)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
