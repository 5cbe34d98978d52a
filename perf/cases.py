"""The work that a user of this framework has it do, as measurable cases.

Three public entry points carry it:

* ``HipKernelLauncher``: one fusion group (GEMM, epilogue chain, optional
  reductions), the callable that the ``torch.compile`` backend binds to a group
  and that an integrator calls directly;
* ``HipMlpLauncher``: a whole MLP block, weights kept packed by its owner;
* ``torch.compile(model, backend=FuseMLCompiler())``: a whole forward under the
  default options, its cost model included.

The framework is for inference, so the directions are decode (a few rows) and
prefill (many rows).  The listed widths are those of ``fuseml_amd/workloads.py``:
its C1-C5 configurations and the reference's presets.  Weights follow
``nn.Linear``'s default initialisation, activations are standard normal.
"""

import math

import torch
import torch.nn as nn

from fuseml_amd.compiler import FuseMLCompiler
from fuseml_amd.epilogue import EpilogueSpec, EpiOp
from fuseml_amd.launcher import HipKernelLauncher
from fuseml_amd.mlp import HipMlpLauncher
from fuseml_amd.workloads import TransformerMLP

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
_DEVICE = "cuda"

# The epilogue chains of the framework's workloads: what follows the GEMM.
# bias_gelu: an MLP's up projection (C2, C5, every preset); bias_gelu_tanh: C1's;
# bias_residual: its down projection; act_heavy: C3; gelu_scale: the activation-
# heavy preset's first GEMM; relu_rows: C4 (its three reductions are per row);
# relu_cols: the same along the other axis.
_CHAINS = ("bias_gelu", "bias_gelu_tanh", "bias_residual", "bias_relu", "act_heavy", "gelu_scale", "relu_rows",
           "relu_cols")


def _group(name, m, n, k, chain, dtype="bf16"):
    return {"name": name, "kind": "group", "M": m, "N": n, "K": k, "chain": chain, "dtype": dtype}


def _block(name, kind, m, d, i, dtype="bf16"):
    return {"name": name, "kind": kind, "M": m, "D": d, "I": i, "dtype": dtype}


def listed():
    return [
        # Decode: a step of a few sequences through an MLP of C2's widths, up
        # projection, and through one of C5's, down projection (long K).
        _group("decode_up", 16, 4096, 1024, "bias_gelu"),
        _group("decode_wide_down", 8, 4096, 16384, "bias_residual"),
        # The smallest configuration (C1): fp32, its first GEMM.
        _group("c1_fp32_up", 64, 2048, 512, "bias_gelu_tanh", "fp32"),
        # The smallest preset as a whole compiled forward.
        _block("small_compiled", "compiled", 128, 256, 1024),
        # A short prefill at the medium preset's widths: the down projection.
        _group("medium_down", 2048, 1024, 4096, "bias_residual"),
        # The preset that runs as a single kernel.
        _block("memory_bound_mlp", "mlp", 16384, 256, 1024),
        # C2's up projection, C3, and C4 (tile and three row reductions).
        _group("c2_up", 16384, 4096, 1024, "bias_gelu"),
        _group("c3_act_heavy", 16384, 4096, 1024, "act_heavy"),
        _group("c4_row_reductions", 8192, 8192, 2048, "relu_rows"),
        # fp16 at a ragged number of rows, the activation-heavy preset's chain.
        _group("fp16_ragged_gelu_scale", 5003, 4096, 1024, "gelu_scale", "fp16"),
        # fp32 prefill at C2's widths.
        _group("fp32_up", 4096, 4096, 1024, "bias_gelu", "fp32"),
        # The largest GEMM: C5's down projection.
        _group("c5_down", 8192, 4096, 16384, "bias_residual"),
    ]


def _log_int(rng, low, high, step=1):
    v = math.exp(rng.uniform(math.log(low), math.log(high)))
    return max(low, int(round(v / step)) * step)


def draw(rng):
    kind = rng.choices(("decode", "group", "fp32", "mlp", "compiled"), (4, 7, 3, 1, 1))[0]
    dtype = rng.choice(("bf16", "bf16", "bf16", "fp16"))
    step = rng.choice((1, 8, 8, 64, 64))  # of the output width: odd ones, as a vocabulary's, among them
    if kind == "mlp":
        return _unnamed(_block("", "mlp", _log_int(rng, 256, 32768), rng.choice((256, 512)), _log_int(rng, 256, 2048, 128),
                               dtype))
    if kind == "compiled":
        return _unnamed(_block("", "compiled", _log_int(rng, 8, 4096), _log_int(rng, 128, 1024, 64),
                               _log_int(rng, 256, 4096, 64), dtype))
    if kind == "decode":
        chain = rng.choice(("bias_gelu", "bias_gelu_tanh", "bias_residual", "bias_relu", "gelu_scale"))
        return _unnamed(_group("", _log_int(rng, 1, 128), _log_int(rng, 256, 16384, step), _log_int(rng, 256, 16384, 8),
                               chain, dtype))
    if kind == "fp32":
        chain = rng.choice(("bias_gelu", "bias_gelu_tanh", "bias_residual", "act_heavy"))
        m, n, k = _log_int(rng, 8, 8192), _log_int(rng, 256, 4096, step), _log_int(rng, 256, 4096)
        while m * n * k > 2 ** 36:
            m = (m + 1) // 2
        return _unnamed(_group("", m, n, k, chain, "fp32"))
    m, n, k = _log_int(rng, 129, 16384), _log_int(rng, 512, 16384, step), _log_int(rng, 256, 8192, 8)
    while m * n * k > 2 ** 38:
        m = (m + 1) // 2
    return _unnamed(_group("", m, n, k, rng.choice(_CHAINS), dtype))


def _unnamed(case):
    del case["name"]
    return case


def _normal(gen, *shape, dtype):
    return torch.randn(*shape, generator=gen, device=_DEVICE).to(dtype)


def _linear(gen, out, inp, dtype):
    """nn.Linear's default initialisation: weight and bias uniform in +-1/sqrt(in)."""
    bound = 1.0 / math.sqrt(inp)

    def uniform(*shape):
        return ((torch.rand(*shape, generator=gen, device=_DEVICE) * 2.0 - 1.0) * bound).to(dtype)

    return uniform(out, inp), uniform(out)


def _spec(chain, dtype):
    """The epilogue of one chain; its inputs are (bias, x, t(W)[, 2-D operand[, row]])."""
    bias, gelu = EpiOp("add", 0), EpiOp("gelu_erf")
    if chain in ("relu_rows", "relu_cols"):
        return EpilogueSpec(0, 1, (EpiOp("relu"),), dtype, reductions=("sum", "amax", "mean"),
                            reduce_axis=1 if chain == "relu_rows" else 0, reduce_dtypes=(torch.float32,) * 3,
                            outputs=(("red", "sum"), ("red", "amax"), ("red", "mean"), ("tile",)))
    ops = {
        "bias_gelu": (bias, gelu),
        "bias_gelu_tanh": (bias, EpiOp("gelu_tanh")),
        "bias_residual": (bias, EpiOp("add", 3)),
        "bias_relu": (bias, EpiOp("relu")),
        "act_heavy": (bias, EpiOp("relu"), EpiOp("mul", 3), EpiOp("sigmoid"), EpiOp("add", 4)),
        "gelu_scale": (bias, gelu, EpiOp("scale", scalar=0.5), EpiOp("add_scalar", scalar=0.125)),
    }[chain]
    return EpilogueSpec(1, 2, ops, dtype)


def _inputs(case, seed):
    """What the case's forward reads, as tensors on the GPU."""
    gen = torch.Generator(device=_DEVICE).manual_seed(seed)
    dtype = _DTYPES[case["dtype"]]
    if case["kind"] != "group":
        M, D, I = case["M"], case["D"], case["I"]
        return (_normal(gen, M, D, dtype=dtype), *_linear(gen, I, D, dtype), *_linear(gen, D, I, dtype))
    M, N, K, chain = case["M"], case["N"], case["K"], case["chain"]
    x = _normal(gen, M, K, dtype=dtype)
    w, b = _linear(gen, N, K, dtype)
    if chain in ("relu_rows", "relu_cols"):
        return x, w.t()
    if chain == "bias_residual":
        return b, x, w.t(), _normal(gen, M, N, dtype=dtype)
    if chain == "act_heavy":  # a gate in [0, 1) and a small row vector, as in C3
        gate = torch.rand(M, N, generator=gen, device=_DEVICE).to(dtype)
        row = ((torch.rand(N, generator=gen, device=_DEVICE) * 2.0 - 1.0) * 0.03).to(dtype)
        return b, x, w.t(), gate, row
    return b, x, w.t()


def prepare(case, seed):
    inputs = _inputs(case, seed)
    if case["kind"] == "group":
        return HipKernelLauncher(_spec(case["chain"], _DTYPES[case["dtype"]]), len(inputs)), inputs
    x, w1, b1, w2, b2 = inputs
    if case["kind"] == "mlp":
        return HipMlpLauncher(), (x, w1.t(), b1, w2.t(), b2, x)
    with torch.device("meta"):
        model = TransformerMLP(case["D"], case["I"])
    for linear, w, b in ((model.linear1, w1, b1), (model.linear2, w2, b2)):
        linear.weight, linear.bias = nn.Parameter(w, requires_grad=False), nn.Parameter(b, requires_grad=False)
    # Every state has a compiled model of its own; Dynamo's default limit of
    # compilations for one forward is meant for one model's changing shapes.
    torch._dynamo.config.recompile_limit = 256
    compiled = torch.compile(model.eval(), backend=FuseMLCompiler(), dynamic=False)
    with torch.no_grad():
        compiled(x)  # compiled at start-up, as a serving program does
    return compiled, (x,)


def run(state):
    fn, inputs = state
    with torch.no_grad():
        return fn(*inputs)


def _size(dtype):
    return 4 if dtype == "fp32" else 2


def work(case):
    e = _size(case["dtype"])
    if case["kind"] != "group":
        M, D, I = case["M"], case["D"], case["I"]
        return {"bytes": float(e * (2 * M * D + 2 * D * I + D + I)), "flops": 4.0 * M * D * I}
    M, N, K, chain = case["M"], case["N"], case["K"], case["chain"]
    elements = M * K + N * K + M * N
    extra = 0
    if chain in ("relu_rows", "relu_cols"):
        extra = 3 * 4 * (M if chain == "relu_rows" else N)
    else:
        elements += N
    if chain in ("bias_residual", "act_heavy"):
        elements += M * N
    if chain == "act_heavy":
        elements += N
    return {"bytes": float(e * elements + extra), "flops": 2.0 * M * N * K}


def tolerance(case):
    # 16-bit results: one rounding of the output (2^-9 for bf16, 2^-12 for fp16,
    # relative, and of the hidden layer in a block).  fp32: a bf16 split product
    # with about 16 mantissa bits and GELU's normal CDF to 1.5e-5.
    if case["dtype"] == "fp32":
        return {"rel": 1e-4, "max": 1e-3}
    if case["dtype"] == "fp16":
        return {"rel": 1e-3, "max": 1e-2}
    return {"rel": 7e-3, "max": 4e-2}


def _gelu(v, tanh=False):
    if tanh:
        return 0.5 * v * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (v + 0.044715 * v ** 3)))
    return 0.5 * v * (1.0 + torch.erf(v / math.sqrt(2.0)))


def exact(case, seed):
    ins = [t.double() for t in _inputs(case, seed)]
    if case["kind"] != "group":
        x, w1, b1, w2, b2 = ins
        return _gelu(x @ w1.t() + b1) @ w2.t() + b2 + x
    chain = case["chain"]
    if chain in ("relu_rows", "relu_cols"):
        v = torch.relu(ins[0] @ ins[1])
        dim = 1 if chain == "relu_rows" else 0
        return v.sum(dim), v.amax(dim), v.mean(dim), v
    b, x, wt = ins[:3]
    v = x @ wt + b
    if chain == "bias_gelu":
        return _gelu(v)
    if chain == "bias_gelu_tanh":
        return _gelu(v, tanh=True)
    if chain == "bias_residual":
        return v + ins[3]
    if chain == "bias_relu":
        return torch.relu(v)
    if chain == "gelu_scale":
        return _gelu(v) * 0.5 + 0.125
    return torch.sigmoid(torch.relu(v) * ins[3]) + ins[4]
