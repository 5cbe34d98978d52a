"""Runtime dispatch of one fused group through the C ABI.

:class:`HipKernelLauncher` keeps the calling convention of the reference's
``KernelLauncher`` (fuseml/codegen/kernel_launcher.py:309-821): it is called
with the group's external tensors positionally, in ``FusionGroup.inputs``
order, has a ``__name__`` for FX node naming (kernel_launcher.py:425-426),
checks arity with ``ValueError`` (685-689), copies negative-stride inputs
(694-703), reads M,K from the left operand and N from the right (709-711),
allocates fresh row-major outputs (723-746), launches on
``torch.cuda.current_stream()`` (622-633) with no host synchronisation, and
returns the primary output — or a tuple ``(primary, *intermediates)`` when the
group has escape outputs, which is what the surgery's ``getitem`` nodes expect
(fuseml/passes/fusion_pass.py:824-880; the reference returns only the primary,
kernel_launcher.py:821).

Instead of ``kernel_fn[grid](ptrs..., M, N, K, strides...)`` it fills a
``fuseml_gemm_desc`` and calls ``fuseml_gemm_epilogue``.  Reductions are
accumulated in fp32 buffers that the library initialises on the stream, then
cast to the reduction's dtype (the reference's fp32-mean path,
kernel_launcher.py:496-509, 816-821, extended to sum and amax).
"""

from __future__ import annotations

import ctypes
import functools
import threading
import warnings
from typing import Any, Callable, Dict, List, Optional, Sequence, Tuple

import torch

from . import _abi
from .epilogue import EpilogueSpec
from .fallback import EagerFallbackGuard

_DTYPE_CODE = {torch.bfloat16: _abi.BF16, torch.float16: _abi.F16, torch.float32: _abi.F32}


def _dtype_code(dt: torch.dtype) -> int:
    try:
        return _DTYPE_CODE[dt]
    except KeyError:
        raise _abi.FuseMLHipError(_abi.EUNSUPPORTED, f"dtype {dt} not supported") from None


def _has_negative_stride(t: torch.Tensor) -> bool:
    return any(s < 0 for s in t.stride())


def _k_major_left(a: torch.Tensor) -> torch.Tensor:
    """A[M,K] with unit K stride, 8-element aligned rows, 16-byte aligned base."""
    if a.stride(1) == 1 and a.stride(0) % 8 == 0 and a.data_ptr() % 16 == 0 and (
        a.stride(0) >= a.shape[1] or a.shape[0] == 1
    ):
        return a
    return a.contiguous()


def _k_major_right(b: torch.Tensor) -> torch.Tensor:
    """B[K,N] with unit K stride (the t(W) view), 8-element aligned columns."""
    if b.stride(0) == 1 and b.stride(1) % 8 == 0 and b.data_ptr() % 16 == 0 and (
        b.stride(1) >= b.shape[0] or b.shape[1] == 1
    ):
        return b
    return b.t().contiguous().t()


def _distinct_bytes(tensors: Sequence[torch.Tensor]) -> int:
    """Bytes of each distinct tensor (by storage span) counted once: what a launch
    must move at least (inputs read once, outputs written once)."""
    seen, total = set(), 0
    for t in tensors:
        if isinstance(t, torch.Tensor):
            key = (t.data_ptr(), t.numel())
            if key not in seen:
                seen.add(key)
                total += t.numel() * t.element_size()
    return total


# 8-byte word index of each pointer / leading-dimension field of the
# descriptor: a call writes them through a flat uint64 view of the structure
# (one C-level store each) instead of through ctypes field accessors.
_WORD = 8
_W_A = _abi.GemmDesc.a.offset // _WORD
_W_LDA = _abi.GemmDesc.lda.offset // _WORD
_W_B = _abi.GemmDesc.b.offset // _WORD
_W_LDB = _abi.GemmDesc.ldb.offset // _WORD
_W_OUT = (_abi.GemmDesc.out.offset + _abi.Output.ptr.offset) // _WORD


def _w_operand(i: int) -> int:
    return (_abi.GemmDesc.operands.offset + i * ctypes.sizeof(_abi.Operand) + _abi.Operand.ptr.offset) // _WORD


def _w_extra(i: int) -> int:
    return (_abi.GemmDesc.extra.offset + i * ctypes.sizeof(_abi.Output) + _abi.Output.ptr.offset) // _WORD


def _w_reduce(slot: int) -> int:
    return _abi.GemmDesc.reduce_out.offset // _WORD + slot


assert all(o % _WORD == 0 for o in (_abi.GemmDesc.a.offset, _abi.GemmDesc.operands.offset,
                                     ctypes.sizeof(_abi.Operand), _abi.GemmDesc.out.offset,
                                     _abi.GemmDesc.extra.offset, ctypes.sizeof(_abi.Output),
                                     _abi.GemmDesc.reduce_out.offset, ctypes.sizeof(_abi.GemmDesc)))


# A signature's calls run in native code after this many: handing a plan over costs
# some microseconds (tens in a process whose caches hold other work), which a
# signature that is seen once or twice would not get back.
_NATIVE_AFTER = 3
_native_lock = threading.Lock()


@functools.lru_cache(maxsize=None)
def _native_type() -> Optional[type]:
    """The native caller's type, or None with a warning where the extension is not
    built, or built for another Python or torch: Python serves every call then."""
    try:
        return _abi.load_fastcall()
    except ImportError as exc:
        warnings.warn(f"repeated launches stay in Python: {exc}", RuntimeWarning)
        return None


class _Plan:
    """What a launch needs that depends only on the input signature (shapes,
    strides, dtypes): the descriptor with every non-pointer field filled, M/N/K,
    and for each operand slot the input it comes from and whether it must be
    rebuilt per call (a dtype conversion or a broadcast that merging copies).

    ``direct``: fp32 operands the library multiplies as they are
    (``fuseml_gemm_epilogue_f32``: a small output, K-major rows); a call whose
    bases are not 16-byte aligned takes ``split_plan``, the same signature's
    plan on split operands.

    ``fast``: a call needs only the pointers (no negative strides, no operand
    rebuilt per call, no fp32 split, a non-empty output); ``a_ok`` / ``b_ok``:
    the GEMM operands' strides are K-major as the kernel reads them (their base
    alignment is still checked per call).

    A call writes its pointers into a descriptor that is its own until the library
    has read it (:meth:`take`: ``desc``, or a copy while another thread's call holds
    that), so threads may share a plan."""

    __slots__ = ("desc", "M", "N", "K", "neg", "operands", "nbytes", "k_split", "fast", "free", "desc_ref",
                 "a_ok", "b_ok", "lda", "ldb", "op_words", "red_words", "extra_words", "single_tile", "direct",
                 "split_plan", "calls", "handed_over")

    def __init__(self) -> None:
        self.desc = _abi.GemmDesc()
        self.M = self.N = self.K = 0
        self.neg = False
        # fp32 GEMM operands: the bf16 segment width k_pad of the three-term
        # split (the kernel then runs K' = 3 k_pad); 0 for bf16/f16 operands.
        self.k_split = 0
        self.operands: List[Tuple[int, bool]] = []  # (input index, rebuilt per call)
        self.nbytes: Optional[int] = None  # algorithmic bytes, for the timing hook
        self.fast = False
        self.desc_ref = ctypes.byref(self.desc)
        # the descriptors that no call is using: as many as calls ran at once
        self.free: List["_CallDesc"] = [_CallDesc(self.desc)]
        self.a_ok = self.b_ok = False
        self.lda = self.ldb = 0
        self.op_words: List[Tuple[int, int]] = []     # (descriptor word, input index)
        self.red_words: List[Tuple[int, str]] = []    # (descriptor word, reduction name)
        self.extra_words: List[int] = []
        self.single_tile = False
        self.direct = False
        self.split_plan: Optional["_Plan"] = None
        self.calls = 0  # fast calls made in Python
        self.handed_over = False  # to the native caller, whether or not it took the plan

    def take(self) -> "_CallDesc":
        """A descriptor for one call, to be put back on ``free`` (both are single
        list operations, which threads may interleave)."""
        try:
            return self.free.pop()
        except IndexError:
            # the fields that the holder of `desc` may be writing are written anew
            return _CallDesc(_abi.GemmDesc.from_buffer_copy(self.desc))


class _CallDesc:
    """A descriptor, also as uint64 words."""

    __slots__ = ("desc", "words", "ref")

    def __init__(self, desc: _abi.GemmDesc) -> None:
        self.desc = desc
        self.words = (ctypes.c_uint64 * (ctypes.sizeof(_abi.GemmDesc) // _WORD)).from_buffer(self.desc)
        self.ref = ctypes.byref(self.desc)


class HipKernelLauncher:
    """Callable that runs one fused group on the gfx950 kernel family."""

    def __init__(
        self,
        spec: EpilogueSpec,
        n_inputs: int,
        eager_fn: Optional[Callable[..., Any]] = None,
        kernel_signature: str = "",
    ) -> None:
        self.__name__ = "fuseml_fused_kernel"
        self.spec = spec
        self._n_inputs = n_inputs
        self._lib = _abi.load_library()
        self._plans: Dict[tuple, _Plan] = {}
        self._fallback_guard: Optional[EagerFallbackGuard] = None
        if eager_fn is not None:
            self._fallback_guard = EagerFallbackGuard(
                eager_fn=eager_fn, kernel_signature=kernel_signature or spec.describe()
            )
        self._python_launches = 0
        # Measurement hook: a list to receive, per launch, (start event, end
        # event, (M, N, K), algorithmic bytes) recorded on the launch stream
        # around the C call.  None (the default) records nothing.  Pairs of
        # timing events taken from `timing_pool` (filled by the caller before
        # a timed region) keep event creation out of that region.
        self.timing_events: Optional[List[Tuple[Any, Any, Tuple[int, int, int], int]]] = None
        self.timing_pool: List[Tuple[Any, Any]] = []
        # Input slots the launch reads: the GEMM operands and the epilogue operands.
        self._used = sorted({spec.left, spec.right} | {op.operand for op in spec.ops if op.kind in ("add", "mul")})
        # Repeated calls of a signature whose plan needs only pointers run in native
        # code (csrc/fastcall.cpp); it declines every other call.
        self._native_type = _native_type()
        self._native: Optional[Any] = None  # made with the first plan handed over
        self._native_call: Optional[Callable[..., Any]] = None

    # ------------------------------------------------------------------
    @property
    def launch_count(self) -> int:
        return self._python_launches + (self._native.count if self._native is not None else 0)

    @launch_count.setter
    def launch_count(self, value: int) -> None:
        self._python_launches = value - (self._native.count if self._native is not None else 0)

    @property
    def fallback_count(self) -> int:
        return self._fallback_guard.fallback_count if self._fallback_guard else 0

    def __repr__(self) -> str:
        return f"HipKernelLauncher({self.spec.describe()})"

    # ------------------------------------------------------------------
    def _operand_tensor(self, t: torch.Tensor, op_index: int, M: int, N: int) -> torch.Tensor:
        """An add/mul operand as a zero-stride-broadcast [M,N] view.

        An operand of an op on an N-D value ([*lead, N], same memory order as
        [M,N]) is broadcast to that shape first and its leading dimensions
        merged; when their strides do not merge (e.g. [B,1,N] against
        [B,S,N]) the merge materialises the broadcast (a copy, still exact).
        """
        if t.dtype not in _DTYPE_CODE:
            t = t.to(torch.float32)
        shape = dict(self.spec.operand_shapes).get(op_index)
        if shape is not None:
            return t.expand(shape).reshape(M, N)
        if t.dim() > 2:
            raise _abi.FuseMLHipError(_abi.EUNSUPPORTED, "operand rank > 2")
        return t.expand(M, N)

    def _operand_order(self) -> List[int]:
        """Input index of each operand slot (first-use order, deduplicated)."""
        order: List[int] = []
        for op in self.spec.ops:
            if op.kind in ("add", "mul") and op.operand not in order:
                order.append(op.operand)
        return order

    def _make_plan(self, inputs: Sequence[torch.Tensor], allow_direct: bool = True) -> _Plan:
        spec = self.spec
        plan = _Plan()
        plan.neg = any(_has_negative_stride(inputs[i]) for i in self._used if isinstance(inputs[i], torch.Tensor))
        if plan.neg:
            inputs = tuple(t.contiguous() if isinstance(t, torch.Tensor) else t for t in inputs)
        a, b = inputs[spec.left], inputs[spec.right]
        if a.dtype != b.dtype or a.dtype not in (torch.bfloat16, torch.float16, torch.float32):
            raise _abi.FuseMLHipError(
                _abi.EUNSUPPORTED, f"GEMM operands {a.dtype}/{b.dtype}: bf16, f16 or fp32 (split) only"
            )
        M, K = int(a.shape[0]), int(a.shape[1])
        N = int(b.shape[1])
        plan.M, plan.N, plan.K = M, N, K
        d = plan.desc
        d.M, d.N, d.K = M, N, K
        if a.dtype == torch.float32:
            # One bf16 GEMM over [hi|hi|lo] . [hi|lo|hi]: K' = 3 k_pad.
            plan.k_split = -(-K // 8) * 8
            d.K = 3 * plan.k_split
            d.ab_dtype = _abi.BF16
        else:
            d.ab_dtype = _dtype_code(a.dtype)
        order = self._operand_order()
        slot = {idx: i for i, idx in enumerate(order)}
        d.n_ops = len(spec.ops)
        if d.n_ops > _abi.MAX_OPS:
            raise _abi.FuseMLHipError(_abi.EUNSUPPORTED, "too many epilogue ops")
        for i, op in enumerate(spec.ops):
            e = d.ops[i]
            e.kind = _abi.OP_CODES[op.kind]
            e.operand = slot[op.operand] if op.kind in ("add", "mul") else op.operand
            e.scalar = op.scalar
        d.n_operands = len(order)
        if d.n_operands > _abi.MAX_OPERANDS:
            raise _abi.FuseMLHipError(_abi.EUNSUPPORTED, "too many epilogue operands")
        for i, idx in enumerate(order):
            src = inputs[idx]
            t = self._operand_tensor(src, idx, M, N)
            o = d.operands[i]
            sm, sn = t.stride()
            o.stride_m, o.stride_n = sm, sn
            o.extent = (M - 1) * sm + (N - 1) * sn + 1
            o.dtype = _DTYPE_CODE[t.dtype]
            # A view of the input itself needs only its pointer per call.
            direct = t.dtype == src.dtype and t.data_ptr() == src.data_ptr() and \
                t.untyped_storage().data_ptr() == src.untyped_storage().data_ptr()
            plan.operands.append((idx, not direct))
        d.out.ld, d.out.dtype = N, _dtype_code(spec.out_dtype) if spec.store_tile else _abi.BF16
        d.n_extra = len(spec.extra_dtypes)
        for i, dt in enumerate(spec.extra_dtypes):
            d.extra[i].ld, d.extra[i].dtype = N, _dtype_code(dt)
        mask = 0
        for name in spec.reductions:
            mask |= _abi.RED_BITS[name]
        d.reduce_mask = mask
        d.reduce_axis = spec.reduce_axis
        # The per-call fast path (see _Plan).
        if not plan.k_split:
            plan.a_ok = a.stride(1) == 1 and a.stride(0) % 8 == 0 and (a.stride(0) >= K or M == 1)
            plan.b_ok = b.stride(0) == 1 and b.stride(1) % 8 == 0 and (b.stride(1) >= K or N == 1)
            plan.lda, plan.ldb = a.stride(0), b.stride(1)
        plan.op_words = [(_w_operand(i), idx) for i, (idx, _) in enumerate(plan.operands)]
        plan.red_words = [(_w_reduce(_abi.RED_SLOT[name]), name) for name in spec.reductions]
        plan.extra_words = [_w_extra(i) for i in range(len(spec.extra_dtypes))]
        plan.single_tile = spec.outputs == (("tile",),) and not spec.output_shapes and spec.store_tile
        ready = not plan.neg and M > 0 and N > 0 and not any(rebuild for _, rebuild in plan.operands)
        if ready and plan.k_split and allow_direct and isinstance(self._lib, ctypes.CDLL):
            self._try_direct(plan, inputs, a, b)
        plan.fast = ready and not plan.k_split
        return plan

    def _try_direct(self, plan: _Plan, inputs: Sequence[torch.Tensor], a: torch.Tensor, b: torch.Tensor) -> None:
        """Turn an fp32 plan into a direct one if the library takes its
        descriptor with the operands as they are."""
        if a.stride(1) != 1 or b.stride(0) != 1:
            return
        probe = _abi.GemmDesc.from_buffer_copy(plan.desc)
        probe.K, probe.ab_dtype, probe.lda, probe.ldb = plan.K, _abi.F32, a.stride(0), b.stride(1)
        # any aligned addresses: the calls' own are checked per call
        probe.a = probe.b = probe.out.ptr = 1 << 12
        for i in range(probe.n_operands):
            probe.operands[i].ptr = 1 << 12
        for i in range(probe.n_extra):
            probe.extra[i].ptr = 1 << 12
        for slot in range(3):
            probe.reduce_out[slot] = 1 << 12
        if not self._lib.fuseml_gemm_epilogue_f32_supported(ctypes.byref(probe)):
            return
        plan.direct = plan.a_ok = plan.b_ok = True
        plan.k_split = 0
        plan.desc.K, plan.desc.ab_dtype = plan.K, _abi.F32
        plan.lda, plan.ldb = a.stride(0), b.stride(1)

    def launch(self, *inputs: torch.Tensor) -> Any:
        """Allocate outputs, set the descriptor's pointers and call the C ABI."""
        spec = self.spec
        key = tuple((t.shape, t.stride(), t.dtype) if isinstance(t, torch.Tensor) else None
                    for t in (inputs[i] for i in self._used))
        plan = self._plans.get(key)
        if plan is None:
            plan = self._plans.setdefault(key, self._make_plan(inputs))
        if plan.direct and (inputs[self.spec.left].data_ptr() | inputs[self.spec.right].data_ptr()) % 16:
            if plan.split_plan is None:
                plan.split_plan = self._make_plan(inputs, allow_direct=False)
            plan = plan.split_plan
        # (tests may bind a recorder as the library: the general path, which
        # assumes no device, serves those)
        if plan.fast and self.timing_events is None and isinstance(self._lib, ctypes.CDLL):
            out = self._launch_fast(plan, inputs)
            plan.calls += 1
            if plan.calls >= _NATIVE_AFTER and not plan.handed_over and plan.a_ok and plan.b_ok:
                # While the GPU works on this call.
                self._add_native(plan, inputs)
            return out
        return self._launch_general(plan, inputs)

    def _add_native(self, plan: _Plan, inputs: Sequence[torch.Tensor]) -> None:
        """Hand a plan whose calls need only pointers to the native caller, unless
        its results are cast or viewed after the launch."""
        spec = self.spec
        with _native_lock:  # once per plan; one caller per launcher: it holds the launch count
            if plan.handed_over:
                return
            plan.handed_over = True
            if self._native_type is None or spec.output_shapes or any(dt is not torch.float32 for dt in spec.reduce_dtypes):
                return
            if self._native is None:
                self._native = self._native_type(self._n_inputs, tuple(self._used), self._fallback_guard is not None)
                self._native_call = self._native.call
        desc = _abi.GemmDesc.from_buffer_copy(plan.desc)
        desc.lda, desc.ldb = plan.lda, plan.ldb
        if plan.single_tile:
            outputs = (("t", 0),)
        else:
            outputs = tuple(("t", 0) if o[0] == "tile" else
                            ("r", spec.reductions.index(o[1])) if o[0] == "red" else ("e", o[1]) for o in spec.outputs)
        self._native.add(inputs, desc, _abi.entry_address(plan.direct), spec.left, spec.right,
                         tuple([(slot, op[0]) for slot, op in enumerate(plan.operands)]),
                         spec.out_dtype if spec.store_tile else None, spec.extra_dtypes,
                         tuple([_abi.RED_SLOT[name] for name in spec.reductions]), outputs)

    def _launch_fast(self, plan: _Plan, inputs: Sequence[torch.Tensor]) -> Any:
        """A call whose plan needs only pointers: the same checks, allocations
        and C call as the general path, with the descriptor written word by
        word."""
        spec = self.spec
        a, b = inputs[spec.left], inputs[spec.right]
        dev = a.get_device()
        if dev < 0 or any(inputs[i].get_device() != dev for i in self._used):
            raise _abi.FuseMLHipError(
                _abi.EINVAL, f"inputs on {sorted({str(inputs[i].device) for i in self._used})}: "
                "every tensor must be on the launch's GPU")
        call = plan.take()
        w = call.words
        pa, pb = a.data_ptr(), b.data_ptr()
        if plan.a_ok and pa % 16 == 0:
            w[_W_LDA] = plan.lda
        else:
            a = _k_major_left(a)
            pa = a.data_ptr()
            w[_W_LDA] = a.stride(0)
        if plan.b_ok and pb % 16 == 0:
            w[_W_LDB] = plan.ldb
        else:
            b = _k_major_right(b)
            pb = b.data_ptr()
            w[_W_LDB] = b.stride(1)
        w[_W_A] = pa
        w[_W_B] = pb
        for wi, idx in plan.op_words:
            w[wi] = inputs[idx].data_ptr()
        device = a.device
        M, N = plan.M, plan.N
        tile = None
        if spec.store_tile:
            tile = torch.empty((M, N), dtype=spec.out_dtype, device=device)
            w[_W_OUT] = tile.data_ptr()
        else:
            w[_W_OUT] = 0
        extras = []
        for wi, dt in zip(plan.extra_words, spec.extra_dtypes):
            t = torch.empty((M, N), dtype=dt, device=device)
            w[wi] = t.data_ptr()
            extras.append(t)
        reds = {}
        if plan.red_words:
            red_len = M if spec.reduce_axis == 1 else N
            for wi, name in plan.red_words:
                t = torch.empty((red_len,), dtype=torch.float32, device=device)
                w[wi] = t.data_ptr()
                reds[name] = t
        entry = self._lib.fuseml_gemm_epilogue_f32 if plan.direct else self._lib.fuseml_gemm_epilogue
        rc = entry(call.ref, torch._C._cuda_getCurrentRawStream(dev))
        plan.free.append(call)
        if rc != _abi.OK:
            raise _abi.FuseMLHipError(rc, _abi.last_error(self._lib))
        self._python_launches += 1
        if plan.single_tile:
            return tile
        return self._assemble(tile, extras, reds)

    def _launch_general(self, plan: _Plan, inputs: Sequence[torch.Tensor]) -> Any:
        spec = self.spec
        if plan.neg:
            inputs = tuple(t.contiguous() if isinstance(t, torch.Tensor) else t for t in inputs)
        M, N = plan.M, plan.N
        a, b = inputs[spec.left], inputs[spec.right]
        dev = a.device
        if isinstance(self._lib, ctypes.CDLL):
            # The kernels dereference every pointer on the GPU: a host tensor or
            # one on another device would fault there.  Raised before any HIP
            # call, as a recoverable error (Triton raises for CPU tensors too).
            if dev.type != "cuda" or any(inputs[i].device != dev for i in self._used):
                raise _abi.FuseMLHipError(
                    _abi.EINVAL, f"inputs on {sorted({str(inputs[i].device) for i in self._used})}: "
                    "every tensor must be on the launch's GPU")
        if not plan.k_split and not plan.direct:
            a, b = _k_major_left(a), _k_major_right(b)

        tile = None
        if spec.store_tile:
            tile = torch.empty((M, N), dtype=spec.out_dtype, device=dev)
        extras = [torch.empty((M, N), dtype=dt, device=dev) for dt in spec.extra_dtypes]
        red_len = M if spec.reduce_axis == 1 else N
        reds = {name: torch.empty((red_len,), dtype=torch.float32, device=dev) for name in spec.reductions}

        if M == 0 or N == 0:
            # No launch.  A reduction over an empty axis follows torch: sum 0,
            # mean NaN, amax raises (IndexError, as torch.amax does).
            reduced_len = N if spec.reduce_axis == 1 else M
            if red_len > 0 and reduced_len == 0:
                if "amax" in reds:
                    raise IndexError("amax(): Expected reduction dim to have non-zero size.")
                for name, t in reds.items():
                    t.fill_(0.0 if name == "sum" else float("nan"))
            return self._assemble(tile, extras, reds)

        call = plan.take()
        d = call.desc
        stream = torch._C._cuda_getCurrentRawStream(dev.index) if dev.type == "cuda" else 0
        if plan.k_split:
            a, b = self._split_operands(plan, a, b, stream)
            d.a, d.lda = a.data_ptr(), a.stride(0)
            d.b, d.ldb = b.data_ptr(), b.stride(0)
        else:
            d.a, d.lda = a.data_ptr(), a.stride(0)
            d.b, d.ldb = b.data_ptr(), b.stride(1)
        rebuilt = []  # operands built for this call, alive until the launch is queued
        for i, (idx, rebuild) in enumerate(plan.operands):
            t = inputs[idx]
            if rebuild:
                t = self._operand_tensor(t, idx, M, N)
                rebuilt.append(t)
            d.operands[i].ptr = t.data_ptr()
        d.out.ptr = tile.data_ptr() if tile is not None else None
        for i, t in enumerate(extras):
            d.extra[i].ptr = t.data_ptr()
        for name, t in reds.items():
            d.reduce_out[_abi.RED_SLOT[name]] = t.data_ptr()

        timing = self.timing_events
        if timing is not None:
            if self.timing_pool:
                ev0, ev1 = self.timing_pool.pop()
            else:
                ev0, ev1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            ev0.record()
        entry = self._lib.fuseml_gemm_epilogue_f32 if plan.direct else self._lib.fuseml_gemm_epilogue
        rc = entry(call.ref, ctypes.c_void_p(stream))
        plan.free.append(call)
        if rc != _abi.OK:
            raise _abi.FuseMLHipError(rc, _abi.last_error(self._lib))
        if timing is not None:
            ev1.record()
            if plan.nbytes is None:
                outs = [t for t in [tile, *extras, *reds.values()] if t is not None]
                plan.nbytes = _distinct_bytes([inputs[i] for i in self._used] + outs)
            timing.append((ev0, ev1, (M, N, plan.K), plan.nbytes))
        self._python_launches += 1
        return self._assemble(tile, extras, reds)

    def _split_operands(self, plan: _Plan, a: torch.Tensor, b: torch.Tensor, stream: int):
        """fp32 GEMM operands as bf16 split parts on the launch stream:
        A3 [M, 3 k_pad] = [hi|hf|lo] of A, B3 [N, 3 k_pad] = [hi|lo|hf] of the
        weight rows (B[k, n] = b[k, n]; hf = hi with inf/NaN written as 0), so
        that A3 . B3^T is the three-term product with inf/NaN only in hi.hi.
        Both are rebuilt on every call (4 bytes read and 6 written per element
        of each operand); caching B3 for a weight would need a reliable signal
        that the weight is unchanged."""
        kp = plan.k_split
        M, N, K = plan.M, plan.N, plan.K
        a3 = torch.empty((M, 3 * kp), dtype=torch.bfloat16, device=a.device)
        b3 = torch.empty((N, 3 * kp), dtype=torch.bfloat16, device=b.device)
        for src, rows, sr, sk, dst, codes in ((a, M, a.stride(0), a.stride(1), a3, _abi.SPLIT_A),
                                              (b, N, b.stride(1), b.stride(0), b3, _abi.SPLIT_B)):
            rc = self._lib.fuseml_split_bf16x3(ctypes.c_void_p(src.data_ptr()), rows, K, sr, sk,
                                               ctypes.c_void_p(dst.data_ptr()), 3 * kp, kp, codes,
                                               ctypes.c_void_p(stream))
            if rc != _abi.OK:
                raise _abi.FuseMLHipError(rc, _abi.last_error(self._lib))
        return a3, b3

    def _assemble(self, tile, extras, reds) -> Any:
        outs = []
        red_dt = dict(zip(self.spec.reductions, self.spec.reduce_dtypes))
        for o in self.spec.outputs:
            if o[0] == "tile":
                outs.append(tile)
            elif o[0] == "red":
                r = reds[o[1]]
                dt = red_dt.get(o[1], torch.float32)
                outs.append(r if dt == torch.float32 else r.to(dt))
            else:
                outs.append(extras[o[1]])
        if self.spec.output_shapes:
            outs = [t if sh is None else t.view(sh) for t, sh in zip(outs, self.spec.output_shapes)]
        return outs[0] if len(outs) == 1 else tuple(outs)

    # ------------------------------------------------------------------
    def __call__(self, *inputs: torch.Tensor) -> Any:
        if self._native_call is not None and self.timing_events is None:
            try:
                out = self._native_call(inputs)
                if type(out) is int:
                    raise _abi.FuseMLHipError(out, _abi.last_error(self._lib))
            except Exception as exc:  # noqa: BLE001 - as the guard filters them
                guard = self._fallback_guard
                if guard is None or not guard.is_recoverable(exc):
                    raise
                return guard.recover(exc, inputs)
            if out is not None:
                return out
        if len(inputs) != self._n_inputs:
            raise ValueError(f"Expected {self._n_inputs} input tensor(s), got {len(inputs)}.")
        if self._fallback_guard is not None:
            return self._fallback_guard.execute(self.launch, inputs)
        return self.launch(*inputs)
