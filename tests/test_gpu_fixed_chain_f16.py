"""The fixed-chain kernels for fp16 operands: bitwise the generic op loop's
results (the same arithmetic on the same values), on whole and ragged tiles and
several rounds; reductions as test_gpu_parity holds the bf16 ones.
"""

from __future__ import annotations

import pytest
import torch

from oracle import gemm_epilogue as ora
from test_gpu_parity import FIXED, _chain_of, _check_tile, _gemm_inputs, _launcher, _np, _operands, _spec

pytestmark = pytest.mark.gpu


def _both(spec, inputs, want):
    from fuseml_amd import _abi

    outs = []
    try:
        for variant, chain in (("deep3", want), ("deep3-generic", 0)):
            _abi.force_variant(variant)
            L = _launcher(spec, len(inputs))
            outs.append(L(*inputs))
            torch.cuda.synchronize()
            assert _chain_of(L) == chain, (variant, _chain_of(L))
    finally:
        _abi.force_variant(None)
    return outs


@pytest.mark.parametrize("name", sorted(FIXED))
@pytest.mark.parametrize("shape", [(600, 1032, 192), (4392, 4360, 128)], ids=lambda s: "x".join(map(str, s)))
def test_fp16_fixed_chain_bitwise_equals_generic(name, shape):
    M, N, K = shape
    dtype = torch.float16
    a, w = _gemm_inputs(M, N, K, dtype, seed=91)
    a[1, :] = a[1, :].sign() * 4e4  # finite operands whose results pass the largest fp16 and saturate
    ops = _operands(M, N, dtype, seed=92)
    host = ops + [a, w.t()]
    left, right = len(ops), len(ops) + 1
    steps, want = FIXED[name]
    print(f"case fp16 fixed chain={name} shape={shape}", flush=True)
    fixed, generic = _both(_spec(left=left, right=right, ops=steps, out_dtype=dtype), [t.cuda() for t in host], want)
    assert torch.equal(fixed, generic), f"{name}: fixed differs from generic"
    ref = ora.gemm_epilogue([_np(t) for t in host], left, right, steps)["tile"].clip(-65504, 65504)
    _check_tile(fixed, ref, f"fp16 fixed {name} {shape}")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("shape", [(600, 1032, 192), (4392, 4360, 128)], ids=lambda s: "x".join(map(str, s)))
def test_gelu_scale_fixed_chain_bitwise_equals_generic(shape, dtype):
    """The activation-heavy block's first group: GELU, then a scale and a scalar
    add, each rounded."""
    M, N, K = shape
    a, w = _gemm_inputs(M, N, K, dtype, seed=96)
    host = [_operands(M, N, dtype, seed=97)[0], a, w.t()]
    steps = [("add", 0, 1.0), ("gelu_erf", -1, 1.0), ("scale", -1, 0.3), ("add_scalar", -1, 0.125)]
    spec = _spec(left=1, right=2, ops=steps, out_dtype=dtype)
    fixed, generic = _both(spec, [t.cuda() for t in host], 9)
    assert torch.equal(fixed, generic)
    _check_tile(fixed, ora.gemm_epilogue([_np(t) for t in host], 1, 2, steps)["tile"])


@pytest.mark.parametrize("axis", [1, 0])
def test_fp16_fixed_relu_reductions_equal_generic(axis):
    dtype = torch.float16
    a, w = _gemm_inputs(600, 1032, 128, dtype, seed=93)
    spec = _spec(left=0, right=1, ops=[("relu", -1, 1.0)], out_dtype=dtype, reductions=("sum", "amax", "mean"),
                 reduce_axis=axis, reduce_dtypes=(torch.float32,) * 3,
                 outputs=(("tile",), ("red", "sum"), ("red", "amax"), ("red", "mean")))
    (ft, fs, fm, fmean), (gt, gs, gm, gmean) = _both(spec, [a.cuda(), w.t().cuda()], 8)
    assert torch.equal(ft, gt) and torch.equal(fm, gm)
    # fp32 atomics add the workgroups' partials in no fixed order
    assert torch.allclose(fs, gs, rtol=1e-6, atol=1e-6) and torch.allclose(fmean, gmean, rtol=1e-6, atol=1e-6)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("chain,k,waves", [("bias_residual", 1024, 4), ("bias_gelu", 1024, 8), ("bias_gelu", 2048, 4)])
def test_partial_round_of_large_tiles(chain, k, waves, dtype):
    """150 tiles of 256x256: the fixed chains run on the one-wave kernel there
    too (GELU(erf) from K = 2048)."""
    import ctypes

    from fuseml_amd import _abi

    M, N = 2500, 3840
    a, w = _gemm_inputs(M, N, k, dtype, seed=94)
    ops = _operands(M, N, dtype, seed=95)[:2]
    host = ops + [a, w.t()]
    L = _launcher(_spec(left=2, right=3, ops=FIXED[chain][0], out_dtype=dtype), 4)
    out = L(*[t.cuda() for t in host])
    (plan,) = L._plans.values()
    cfg = (ctypes.c_int32 * 4)()
    assert _abi.load_library().fuseml_gemm_epilogue_config(plan.desc_ref, cfg) == 0
    assert tuple(cfg[:3]) == (256, 256, waves)
    rows = [0, 255, 256, 1000, M - 1]
    host[1], host[2] = host[1][rows], host[2][rows]
    ref = ora.gemm_epilogue([_np(t) for t in host], 2, 3, FIXED[chain][0])["tile"]
    _check_tile(out[rows], ref, f"{chain} {k}")
