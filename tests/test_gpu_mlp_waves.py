"""The eight-wave single-kernel MLP (packed weights) at the edges of its row
blocks and super-chunks: bitwise the four-wave kernel on unpacked weights (the
same products summed in the same order), and close to the oracle.
"""

from __future__ import annotations

import pytest
import torch

from test_gpu_mlp_block import _close, _inputs, _oracle

pytestmark = pytest.mark.gpu


# 32-row blocks up to 32 rows per CU (8192 on 256 CUs), 64-row ones above; more
# rows than one block per CU; I of one super-chunk, half of one, and a half last.
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("shape", [(1, 256, 128), (33, 512, 128), (31, 256, 384), (8192, 256, 256), (8193, 256, 640),
                                   (8225, 512, 256), (16421, 256, 256), (300, 512, 1152)],
                         ids=lambda s: "x".join(map(str, s)))
def test_packed_equals_unpacked(shape, dtype):
    from fuseml_amd.mlp import HipMlpLauncher

    M, D, I = shape
    x, w1, b1, w2, b2, r = _inputs(M, D, I, dtype, seed=5)
    args = (x.cuda(), w1.cuda().t(), b1.cuda(), w2.cuda().t(), b2.cuda(), r.cuda())
    print(f"case mlp waves {shape} {dtype}", flush=True)
    for approximate, post in (("none", ()), ("tanh", (("scale", 0.5), ("add_scalar", 0.125)))):
        got = HipMlpLauncher(approximate, post=post)(*args)
        want = HipMlpLauncher(approximate, post=post, pack_weights=False)(*args)
        torch.cuda.synchronize()
        assert torch.equal(got, want)
    rows = sorted({0, M // 2, M - 1})
    y = HipMlpLauncher()(*args)
    _close(y[rows], _oracle(x[rows], w1, b1, w2, b2, r[rows]), f"{shape}")


def test_strided_rows_and_missing_terms():
    """x, r and y rows with their own pitch; no b2, no residual."""
    from fuseml_amd.mlp import HipMlpLauncher

    M, D, I = 100, 256, 384
    x, w1, b1, w2, b2, r = _inputs(M, D, I, torch.bfloat16, seed=6)
    wide = torch.zeros(M, D + 8, dtype=x.dtype).cuda()
    wide[:, :D] = x.cuda()
    base = (w1.cuda().t(), b1.cuda(), w2.cuda().t())
    for b, res in ((None, None), (b2.cuda(), None), (None, wide[:, :D])):
        args = (wide[:, :D], *base, b, res)
        assert torch.equal(HipMlpLauncher()(*args), HipMlpLauncher(pack_weights=False)(*args))
