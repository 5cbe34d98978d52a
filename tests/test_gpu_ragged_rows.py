"""Rows that are not whole 16-byte chunks at 16-byte addresses (any N, any row
stride, any 2-byte aligned base), staged in LDS like the others: against the
CPU oracle on every tile variant, and nothing written outside the rows.  And
column reductions beside a staged output and a staged 2-D operand.
"""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from oracle import gemm_epilogue as ora
from test_gpu_parity import CHAINS, _check_red, _check_tile, _gemm_inputs, _gen, _launcher, _np, _operands, _spec

pytestmark = pytest.mark.gpu

VARIANTS = ["large", "deep3", "deep", "large128", "small", "small64", "narrow64", "narrow32"]


@pytest.fixture(params=VARIANTS)
def variant(request):
    from fuseml_amd import _abi

    _abi.force_variant(request.param)
    yield request.param
    _abi.force_variant(None)


def _residual_views(M, N, dtype):
    """[M, N] operands of every row alignment: odd row stride, a column offset
    of 1 to 8 elements, the end of a storage."""
    g = _gen(3)
    wide = torch.randn(M, N + 9, generator=g).to(dtype).cuda()
    flat = torch.randn(M * N + 5, generator=g).to(dtype).cuda()
    return {"contiguous": wide[:, :N].contiguous(), "offset1": wide[:, 1:1 + N], "offset8": wide[:, 8:8 + N],
            "end": flat[5:].view(M, N)}


@pytest.mark.parametrize("n", [8, 9, 15, 257, 1030, 1031, 516])
def test_ragged_rows_parity(variant, n):
    M, K, dtype = 270, 128, torch.bfloat16
    a, w = _gemm_inputs(M, n, K, dtype, seed=61)
    bias = _operands(M, n, dtype, seed=62)[0]
    steps = [("add", 0, 1.0), ("add", 1, 0.5), ("relu", -1, 1.0)]
    for what, r in _residual_views(M, n, dtype).items():
        print(f"case ragged rows {variant} N={n} {what}", flush=True)
        inputs = [bias.cuda(), r, a.cuda(), w.t().cuda()]
        L = _launcher(_spec(left=2, right=3, ops=steps, out_dtype=dtype), 4)
        out = L(*inputs)
        torch.cuda.synchronize()
        _check_tile(out, ora.gemm_epilogue([_np(t) for t in inputs], 2, 3, steps)["tile"], f"{variant} {n} {what}")


@pytest.mark.parametrize("n,ld,offset", [(1031, 1031, 0), (1031, 1040, 1), (264, 265, 3), (264, 264, 1), (13, 14, 1)])
def test_only_the_rows_are_written(variant, n, ld, offset):
    """Through the C ABI: an output with its own row stride and base offset, in a
    buffer of a known pattern; every byte outside the M rows of N keeps it."""
    from fuseml_amd import _abi

    lib = _abi.load_library()
    M, K = 270, 64
    a, w = _gemm_inputs(M, n, K, torch.bfloat16, seed=63)
    da, dw = a.cuda(), w.cuda()
    buf = torch.full((offset + M * ld + 16,), 0x7777, dtype=torch.int16, device="cuda")
    d = _abi.GemmDesc()
    d.M, d.N, d.K, d.ab_dtype = M, n, K, _abi.BF16
    d.a, d.lda, d.b, d.ldb = da.data_ptr(), K, dw.data_ptr(), K
    d.out.ptr, d.out.ld, d.out.dtype = buf.data_ptr() + 2 * offset, ld, _abi.BF16
    print(f"case rows written {variant} {n} {ld} {offset}", flush=True)
    assert lib.fuseml_gemm_epilogue(ctypes.byref(d), torch.cuda.current_stream().cuda_stream) == 0, _abi.last_error(lib)
    torch.cuda.synchronize()
    rows = buf[offset:offset + M * ld].view(M, ld)
    _check_tile(rows[:, :n].view(torch.bfloat16), _np(a) @ _np(w).T)
    assert (rows[:, n:] == 0x7777).all() and (buf[:offset] == 0x7777).all() and (buf[offset + M * ld:] == 0x7777).all()


@pytest.mark.parametrize("shape", [(600, 1024, 192), (530, 1031, 128), (256, 256, 64), (70, 130, 72)],
                         ids=lambda s: "x".join(map(str, s)))
def test_column_reductions_with_staged_tiles(variant, shape):
    M, N, K = shape
    dtype = torch.bfloat16
    a, w = _gemm_inputs(M, N, K, dtype, seed=65)
    ops = _operands(M, N, dtype, seed=66)[:2]
    inputs = ops + [a, w.t()]
    steps = [("add", 0, 1.0), ("add", 1, 1.0), ("sigmoid", -1, 1.0)]  # sigmoid(0) = 0.5 shows padded elements
    spec = _spec(left=2, right=3, ops=steps, out_dtype=dtype, reductions=("sum", "amax", "mean"), reduce_axis=0,
                 reduce_dtypes=(torch.float32,) * 3,
                 outputs=(("tile",), ("red", "sum"), ("red", "amax"), ("red", "mean")))
    print(f"case column reductions {variant} {shape}", flush=True)
    tile, s, mx, mean = _launcher(spec, 4)(*[t.cuda() for t in inputs])
    torch.cuda.synchronize()
    ref = ora.gemm_epilogue([_np(t) for t in inputs], 2, 3, steps, ("sum", "amax", "mean"), 0)
    v = ref["tile"]
    _check_tile(tile, v)
    _check_red(s, ref["sum"], np.abs(v).sum(axis=0), "sum")
    _check_red(mx, ref["amax"], np.abs(v).max(axis=0), "amax")
    _check_red(mean, ref["mean"], np.abs(v).mean(axis=0), "mean")
    # tighter than the contract's 1e-2: fp32 sums of M values
    assert np.allclose(_np(s), ref["sum"], rtol=1e-4)


@pytest.mark.parametrize("out", ["bf16", "fp32", "none"])
@pytest.mark.parametrize("first,second", [("contiguous", "contiguous"), ("contiguous", "offset1"), ("offset1", "contiguous")])
def test_aligned_and_ragged_launches(variant, first, second, out):
    """Two 2-D operands, each aligned or not, beside a staged output, one that is not
    staged and none (an escape store and a reduction instead): the kernel without the
    code for ragged rows runs where nothing needs it, and only there."""
    M, N, K, dtype = 150, 264, 72, torch.bfloat16
    a, w = _gemm_inputs(M, N, K, dtype, seed=67)
    views = _residual_views(M, N, dtype)
    inputs = [views[first], views[second], a.cuda(), w.t().cuda()]
    steps = [("add", 0, 1.0), ("mul", 1, 1.0), ("relu", -1, 1.0)]
    print(f"case aligned and ragged {variant} {first} {second} {out}", flush=True)
    spec = dict(left=2, right=3, ops=steps, out_dtype=torch.float32 if out == "fp32" else dtype, reductions=("sum",),
                reduce_axis=1, reduce_dtypes=(torch.float32,), outputs=(("tile",), ("red", "sum")))
    if out == "none":
        spec |= dict(ops=steps[:2] + [("store", 0, 1.0)] + steps[2:], store_tile=False, extra_dtypes=(dtype,),
                     outputs=(("extra", 0), ("red", "sum")))
    tile, s = _launcher(_spec(**spec), 4)(*inputs)
    torch.cuda.synchronize()
    values = [_np(t) for t in inputs]
    ref = ora.gemm_epilogue(values, 2, 3, steps, ("sum",), 1)
    _check_tile(tile, ora.gemm_epilogue(values, 2, 3, steps[:2])["tile"] if out == "none" else ref["tile"])
    _check_red(s, ref["sum"], np.abs(ref["tile"]).sum(axis=1), "sum")
