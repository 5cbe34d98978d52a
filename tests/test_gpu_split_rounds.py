"""Outputs of a little more than whole rounds of 256x256 tiles: the rows (or
columns) past the rounds run as a second launch.  Against the same group on one
pinned tile variant and the CPU oracle on rows around the seam; two launches are
asserted by counting them.
"""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from oracle import gemm_epilogue as ora
from test_gpu_parity import _check_tile, _gemm_inputs, _gen, _launcher, _np, _operands, _spec

pytestmark = pytest.mark.gpu

# rows: 16 or 17 tiles of rows in the first part; columns: 512 rows, 128 tiles of columns
CASES = [((4096 + 37, 4096, 192), "rows"), ((4352, 3841, 128), "rows"), ((300, 33000, 136), "cols"),
         ((512, 32768 + 520, 64), "cols")]


def _kernels(fn):
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        fn()
        torch.cuda.synchronize()
    return [e.key for e in prof.key_averages() for _ in range(e.count) if "gemm_" in e.key]


def _run(spec, inputs, pinned=None):
    from fuseml_amd import _abi

    try:
        _abi.force_variant(pinned)
        out = _launcher(spec, len(inputs))(*inputs)
        torch.cuda.synchronize()
        return out
    finally:
        _abi.force_variant(None)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("shape,axis", CASES, ids=lambda v: v if isinstance(v, str) else "x".join(map(str, v)))
def test_split_rounds_parity(shape, axis, dtype):
    M, N, K = shape
    a, w = _gemm_inputs(M, N, K, dtype, seed=71)
    ops = _operands(M, N, dtype, seed=72)
    host = ops + [a, w.t()]
    steps = [("add", 0, 1.0), ("mul", 1, 1.0), ("relu", -1, 1.0), ("add", 2, 1.0), ("add", 3, -0.5)]
    spec = _spec(left=5, right=6, ops=steps, out_dtype=dtype)
    inputs = [t.cuda() for t in host]
    print(f"case split rounds {shape} {dtype}", flush=True)
    got = _run(spec, inputs)
    # fp32 sums in another order: one rounding of the output apart
    torch.testing.assert_close(got.float(), _run(spec, inputs, "large").float(), rtol=2 ** -7, atol=2 ** -7)
    rows = sorted({0, 255, min(4095, M - 1), min(4096, M - 1), M - 1})
    host[1], host[3], host[5] = host[1][rows], host[3][rows], host[5][rows]
    _check_tile(got[rows], ora.gemm_epilogue([_np(t) for t in host], 5, 6, steps)["tile"])


def test_two_launches():
    M, N, K = 4096 + 37, 4096, 192
    a, w = _gemm_inputs(M, N, K, torch.bfloat16, seed=73)
    L = _launcher(_spec(left=0, right=1, ops=[("relu", -1, 1.0)], out_dtype=torch.bfloat16), 2)
    x, wt = a.cuda(), w.cuda().t()
    L(x, wt)
    torch.cuda.synchronize()
    assert len(_kernels(lambda: L(x, wt))) == 2
    assert len(_kernels(lambda: L(x[:4096], wt))) == 1


@pytest.mark.parametrize("shape,axis", CASES, ids=lambda v: v if isinstance(v, str) else "x".join(map(str, v)))
@pytest.mark.parametrize("red_axis", [1, 0])
@pytest.mark.parametrize("reductions", [("sum", "amax"), ("sum", "amax", "mean")], ids="+".join)
def test_split_rounds_reductions(shape, axis, red_axis, reductions):
    """Sums and maxima of both parts meet in one buffer; a mean along the split
    axis keeps one launch (its divisor is the whole length)."""
    M, N, K = shape
    dtype = torch.bfloat16
    a, w = _gemm_inputs(M, N, K, dtype, seed=74)
    x, wt = a.cuda(), w.cuda().t()
    spec = _spec(left=0, right=1, ops=[("sigmoid", -1, 1.0), ("store", 0)], out_dtype=dtype, store_tile=False,
                 extra_dtypes=(torch.float32,), reductions=reductions, reduce_axis=red_axis,
                 reduce_dtypes=(torch.float32,) * len(reductions),
                 outputs=tuple(("red", r) for r in reductions) + (("extra", 0),))
    *reds, tile = _run(spec, [x, wt])
    v = tile.double()
    want = {"sum": v.sum(red_axis), "amax": v.amax(red_axis), "mean": v.mean(red_axis)}
    for r, got in zip(reductions, reds):
        torch.testing.assert_close(got.double(), want[r], rtol=2e-5, atol=1e-6)
    ref = torch.sigmoid(x[:64].double() @ wt.double())
    torch.testing.assert_close(v[:64], ref, rtol=1e-4, atol=1e-4)
