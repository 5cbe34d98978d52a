"""Infinite activations through the single-kernel MLP on packed weights where I is
an odd multiple of 128: its last super-chunk is half one, and no product beyond I
may enter (inf * 0 is NaN).  The unpacked kernel has no columns beyond I.  And the
packed weights are W1 and W2 and no more, on the host and as written.
"""

from __future__ import annotations

import ctypes

import pytest
import torch

from fuseml_amd import _abi

gpu = pytest.mark.gpu


def _desc(D, I, M=64):
    """A descriptor of aligned placeholder addresses (no kernel reads them here)."""
    d = _abi.MlpDesc()
    d.M, d.D, d.I = M, D, I
    d.x = d.w1 = d.b1 = d.w2 = d.y = 1 << 12
    d.ldx = d.ldw1 = d.ldy = D
    d.ldr, d.ldw2 = D, I
    d.dtype, d.gelu = _abi.BF16, _abi.OP_GELU_ERF
    return d


@pytest.mark.parametrize("D", [256, 512])
@pytest.mark.parametrize("I", [128, 256, 384, 1024, 1152])
def test_packed_weights_are_as_large_as_the_weights(D, I):
    """4 D I bytes, as the header states: a caller may size its buffer by that."""
    assert _abi.load_library().fuseml_mlp_pack_bytes(ctypes.byref(_desc(D, I))) == 4 * D * I


@gpu
@pytest.mark.parametrize("shape", [(256, 128), (256, 640), (512, 384), (512, 512)], ids=lambda s: "x".join(map(str, s)))
def test_packing_permutes_the_weights(shape):
    """Every weight exactly once, and nothing written past the stated size."""
    D, I = shape
    w1 = torch.arange(D * I, dtype=torch.int32).view(I, D)
    w2 = (torch.arange(D * I, dtype=torch.int32) + 1).view(D, I)
    w1, w2 = (t.to(torch.int16).cuda() for t in (w1, w2))
    lib = _abi.load_library()
    d = _desc(D, I)
    d.w1, d.w2 = w1.data_ptr(), w2.data_ptr()
    n = lib.fuseml_mlp_pack_bytes(ctypes.byref(d))
    buf = torch.full((n // 2 + 32768,), 12345, dtype=torch.int16, device="cuda")
    print(f"case mlp pack {shape}", flush=True)
    assert lib.fuseml_mlp_pack_weights(ctypes.byref(d), ctypes.c_void_p(buf.data_ptr()),
                                       ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == _abi.OK
    torch.cuda.synchronize()
    assert (buf[n // 2:] == 12345).all()
    want = torch.cat([w1.flatten(), w2.flatten()])
    assert torch.equal(buf[:n // 2].sort().values, want.sort().values)


@gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("sign", [1.0, -1.0], ids=["+inf", "-inf"])
@pytest.mark.parametrize("shape", [(40, 256, 128), (40, 512, 384), (8200, 256, 640), (40, 256, 256)],
                         ids=lambda s: "x".join(map(str, s)))
def test_infinite_rows_stay_as_the_unpacked_kernel_has_them(shape, sign, dtype):
    from fuseml_amd.mlp import HipMlpLauncher

    M, D, I = shape
    g = torch.Generator().manual_seed(I)
    x = torch.randn(M, D, generator=g)
    rows = (0, 33, M - 1)
    x[rows, (0, 5, D - 1)] = sign * float("inf")
    # Positive weights: every sum that has one infinite term is that infinity.
    w1 = torch.rand(I, D, generator=g) / D + 1e-3
    w2 = torch.rand(D, I, generator=g) / I + 1e-3
    b1, b2, r = torch.randn(I, generator=g), torch.randn(D, generator=g), torch.randn(M, D, generator=g)
    x, w1, b1, w2, b2, r = (t.to("cuda", dtype) for t in (x, w1, b1, w2, b2, r))
    args = (x, w1.t(), b1, w2.t(), b2, r)
    print(f"case mlp infinite {shape} {sign} {dtype}", flush=True)
    for approximate, post in (("none", ()), ("tanh", ()), ("none", (("scale", 0.5), ("add_scalar", 0.125)))):
        got = HipMlpLauncher(approximate, post=post)(*args)
        want = HipMlpLauncher(approximate, post=post, pack_weights=False)(*args)
        torch.cuda.synchronize()
        torch.testing.assert_close(got, want, rtol=0, atol=0, equal_nan=True)
        finite = torch.ones(M, dtype=torch.bool)
        finite[list(rows)] = False
        assert torch.isfinite(got.cpu()[finite]).all()
        if sign > 0:  # GELU(+inf) is +inf: no NaN (tanh's -inf * 0 is one, in both kernels)
            assert not torch.isnan(got).any()
