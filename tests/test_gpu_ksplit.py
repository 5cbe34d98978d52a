"""The K-split kernel (small outputs) against the CPU oracle: every tile it
picks, ragged rows, columns and K (ends of a 16-row block, of a 4-column run, of
a 128-byte chunk, fewer chunks than waves), every operand and output form, both
reduction axes.  The route is asserted through fuseml_gemm_epilogue_ksplit.
Tolerances as in test_gpu_parity.
"""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from oracle import gemm_epilogue as ora
from test_gpu_parity import CHAINS, _check_red, _check_tile, _gemm_inputs, _gen, _launcher, _np, _operands, _spec

pytestmark = pytest.mark.gpu

# (M, N, K), (BM, BN, waves)
SHAPES = [
    ((1, 8, 8), (16, 32, 4)),           # one partial chunk, three waves without one
    ((17, 1030, 1000), (16, 32, 4)),    # N % 4 != 0, K ends inside a chunk
    ((100, 257, 4640), (16, 16, 8)),    # odd N
    ((16, 256, 72), (16, 32, 4)),
    ((128, 256, 1024), (16, 32, 4)),    # the reference's small preset's second GEMM
    ((90, 1355, 2312), (32, 16, 4)),
    ((500, 507, 520), (32, 32, 4)),
    ((255, 1001, 1032), (32, 32, 4)),
    ((8, 16384, 1544), (16, 64, 4)),
    ((500, 1023, 2056), (32, 64, 4)),
    ((950, 530, 2056), (64, 32, 4)),
]
_ID = lambda v: "x".join(map(str, v))  # noqa: E731


def _route(L):
    from fuseml_amd import _abi

    (plan,) = L._plans.values()
    cfg = (ctypes.c_int32 * 4)()
    rc = _abi.load_library().fuseml_gemm_epilogue_ksplit(plan.desc_ref, cfg)
    assert rc == 1, (rc, _abi.last_error())
    return tuple(cfg[:3])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("chain", ["bias_gelu", "act_heavy", "scalars", "col_bias_alpha", "bcast_mul"])
@pytest.mark.parametrize("shape,tile", SHAPES, ids=_ID)
def test_ksplit_chain_parity(shape, tile, chain, dtype):
    M, N, K = shape
    a, w = _gemm_inputs(M, N, K, dtype, seed=41)
    ops = _operands(M, N, dtype, seed=42)
    inputs = ops + [a, w.t()]
    left, right = len(ops), len(ops) + 1
    print(f"case ksplit {shape} {chain} {dtype}", flush=True)
    L = _launcher(_spec(left=left, right=right, ops=CHAINS[chain], out_dtype=dtype), len(inputs))
    out = L(*[t.cuda() for t in inputs])
    torch.cuda.synchronize()
    assert _route(L) == tile
    _check_tile(out, ora.gemm_epilogue([_np(t) for t in inputs], left, right, CHAINS[chain])["tile"], f"{chain} {shape}")


@pytest.mark.parametrize("axis", [1, 0])
@pytest.mark.parametrize("shape,tile", SHAPES, ids=_ID)
def test_ksplit_reductions_and_escape(shape, tile, axis):
    """Tile, an escape store of the pre-activation, and three reductions;
    sigmoid(0) = 0.5 would show a padded element in a sum."""
    M, N, K = shape
    dtype = torch.bfloat16
    a, w = _gemm_inputs(M, N, K, dtype, seed=43)
    bias = (torch.rand(N, generator=_gen(5)) - 0.5).to(dtype)
    inputs = [bias, a, w.t()]
    steps = [("add", 0, 1.0), ("sigmoid", -1, 1.0)]
    spec = _spec(left=1, right=2, ops=[steps[0], ("store", 0), steps[1]], out_dtype=dtype, extra_dtypes=(torch.float32,),
                 reductions=("sum", "amax", "mean"), reduce_axis=axis, reduce_dtypes=(torch.float32,) * 3,
                 outputs=(("tile",), ("extra", 0), ("red", "sum"), ("red", "amax"), ("red", "mean")))
    print(f"case ksplit reductions {shape} axis={axis}", flush=True)
    L = _launcher(spec, 3)
    tile_out, pre, s, mx, mean = L(*[t.cuda() for t in inputs])
    torch.cuda.synchronize()
    assert _route(L) == tile
    ins = [_np(t) for t in inputs]
    ref = ora.gemm_epilogue(ins, 1, 2, steps, ("sum", "amax", "mean"), axis)
    v = ref["tile"]
    _check_tile(tile_out, v)
    _check_tile(pre, ora.gemm_epilogue(ins, 1, 2, steps[:1])["tile"], "escape")
    _check_red(s, ref["sum"], np.abs(v).sum(axis=axis), "sum")
    _check_red(mx, ref["amax"], np.abs(v).max(axis=axis), "amax")
    _check_red(mean, ref["mean"], np.abs(v).mean(axis=axis), "mean")


def test_ksplit_layouts_agree_with_the_tiled_kernels():
    """Row-strided, transposed and misaligned operands (an x whose rows are a
    slice, a right operand that has to be copied to K-major): the K-split kernel
    and a pinned tiled variant agree to the rounding of the output, at a
    tolerance of two bf16 units (their fp32 sums differ in order only)."""
    from fuseml_amd import _abi

    M, N, K = 40, 264, 512
    g = _gen(7)
    wide = torch.randn(M, K + 24, generator=g).bfloat16().cuda()
    w = (torch.randn(N, K, generator=g) / K ** 0.5).bfloat16().cuda()
    tile = torch.randn(N, M, generator=g).bfloat16().cuda().t()  # column-major residual
    bias = torch.randn(2 * N, generator=g).bfloat16().cuda()[::2]
    for x in (wide[:, :K], wide[:, 8:8 + K], wide[:, 3:3 + K], wide[::2][:20, :K].repeat(2, 1)):
        for wt in (w.t(), w.t().contiguous()):
            spec = _spec(left=1, right=2, ops=[("add", 0, 1.0), ("add", 3, 0.5), ("relu", -1, 1.0)],
                         out_dtype=torch.bfloat16)
            L = _launcher(spec, 4)
            got = L(bias, x, wt, tile)
            try:
                _abi.force_variant("narrow32")
                want = L(bias, x, wt, tile)
            finally:
                _abi.force_variant(None)
            torch.testing.assert_close(got.float(), want.float(), rtol=2 ** -7, atol=2 ** -7)


# fp32 operands multiplied as they are.
F32_SHAPES = [(1, 8, 4), (64, 2048, 512), (17, 1030, 1004), (33, 257, 36), (31, 4099, 260), (500, 1023, 132),
              (1000, 520, 516)]


@pytest.mark.parametrize("chain", ["bias_gelu_tanh", "act_heavy", "scalars"])
@pytest.mark.parametrize("shape", F32_SHAPES, ids=_ID)
def test_fp32_direct_parity(shape, chain):
    """Against the float64 oracle (1e-4, as every fp32 group), and no further
    from it than the split passes' result of the same inputs: the same bf16
    products, summed in fp32 in another order (1.5x, or 1e-6 of the result)."""
    M, N, K = shape
    a, w = _gemm_inputs(M, N, K, torch.float32, seed=51)
    ops = _operands(M, N, torch.float32, seed=52)
    inputs = ops + [a, w.t()]
    left, right = len(ops), len(ops) + 1
    print(f"case fp32 direct {shape} {chain}", flush=True)
    L = _launcher(_spec(left=left, right=right, ops=CHAINS[chain], out_dtype=torch.float32), len(inputs))
    dev = [t.cuda() for t in inputs]
    got = _np(L(*dev))
    (plan,) = L._plans.values()
    assert plan.direct
    # a base that is not 16-byte aligned takes the split passes
    odd = torch.empty(M * K + 1, device="cuda")[1:].view(M, K).copy_(dev[left])
    split = _np(L(*dev[:left], odd, dev[right]))
    assert plan.split_plan is not None and not plan.split_plan.direct
    ref = ora.gemm_epilogue([_np(t) for t in inputs], left, right, CHAINS[chain])["tile"]
    assert np.isclose(got, ref, rtol=1e-4, atol=1e-4).all(), np.abs(got - ref).max()
    norm = np.linalg.norm(ref)
    assert np.linalg.norm(got - ref) <= 1.5 * np.linalg.norm(split - ref) + 1e-6 * norm


def test_fp32_direct_non_finite_matches_the_split_passes():
    """inf, NaN and values above the largest bf16 in both operands: NaN and inf
    come out where the split passes put them, all else agrees to 1e-4."""
    M, N, K = 40, 72, 100
    a, w = _gemm_inputs(M, N, K, torch.float32, seed=53)
    a[:, ::2] = torch.round(a[:, ::2] * 4) / 4 + 0.25
    a[0, 1], a[3, K - 1], a[5, 50], a[7, 2] = float("inf"), -float("inf"), float("nan"), 3.4e38
    w[2, 3], w[9, 1], w[11, 99] = float("inf"), float("nan"), -3.39e38
    dev, wt = a.cuda(), w.cuda().t()
    L = _launcher(_spec(left=0, right=1, ops=[("scale", -1, 0.5)], out_dtype=torch.float32), 2)
    got = L(dev, wt)
    (plan,) = L._plans.values()
    assert plan.direct
    want = L(torch.empty(M * K + 1, device="cuda")[1:].view(M, K).copy_(dev), wt)
    torch.testing.assert_close(got, want, rtol=1e-4, atol=1e-4, equal_nan=True)
    assert torch.isnan(got).any() and torch.isinf(got).any()
