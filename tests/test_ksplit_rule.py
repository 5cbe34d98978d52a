"""The K-split kernel's rules, compiled from the library's own header on the host:
a probe without a device (256 CUs assumed) and a launch on a device of another CU
count take the same fp32 groups, and the probe is the built library's.
"""

from __future__ import annotations

import ctypes
import pathlib
import random
import shutil
import subprocess

import pytest

from fuseml_amd import _abi

HEADER_DIR = pathlib.Path(__file__).resolve().parents[1] / "fuseml_amd" / "csrc"


@pytest.fixture(scope="module")
def tile(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    d = tmp_path_factory.mktemp("ksplit")
    src, lib = d / "shim.cpp", d / "libksplit.so"
    src.write_text('#include "ksplit_rule.h"\nextern "C" int tile(int64_t m, int64_t n, int64_t k, int cus) '
                   "{ return fuseml_gemm::ksplit_f32(m, n, k, cus); }\n")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", f"-I{HEADER_DIR}", str(src), "-o", str(lib)], check=True)
    so = ctypes.CDLL(str(lib))
    so.tile.argtypes = [ctypes.c_int64] * 3 + [ctypes.c_int]
    return so.tile


def _sizes():
    rng = random.Random(11)
    for _ in range(4000):
        # around the limits of 2^20 and 2^21 elements, ragged
        K = rng.choice((64, 256, 512, 516, 1024, 4096, 16384))
        M = rng.randrange(1, 4097)
        N = max(1, int(rng.uniform(0.5, 1.3) * (1 << (21 if K <= 512 else 20)) / M))
        yield M, N, K


def test_which_sizes_are_taken_does_not_depend_on_the_device(tile):
    taken = [tile(*s, 256) >= 0 for s in _sizes()]
    assert 0.2 < sum(taken) / len(taken) < 0.9
    for cus in (8, 32, 64, 128, 304):
        assert [tile(*s, cus) >= 0 for s in _sizes()] == taken


def test_the_library_takes_what_the_rule_takes(tile):
    lib = _abi.load_library()
    for M, N, K in list(_sizes())[:500]:
        d = _abi.GemmDesc()
        d.M, d.N, d.K = M, N, K
        d.a = d.b = d.out.ptr = 1 << 12
        d.lda = d.ldb = K
        d.ab_dtype = d.out.dtype = _abi.F32
        d.out.ld = N
        assert bool(lib.fuseml_gemm_epilogue_f32_supported(ctypes.byref(d))) == (tile(M, N, K, 256) >= 0)


def test_empty_k_is_not_taken(tile):
    assert tile(16, 16, 0, 256) == -1


def _route(M, N, K, row_reductions=False):
    d = _abi.GemmDesc()
    d.M, d.N, d.K = M, N, K
    d.a = d.b = d.out.ptr = 1 << 12
    d.lda = d.ldb = K
    d.ab_dtype = d.out.dtype = _abi.BF16
    d.out.ld = N
    if row_reductions:
        d.reduce_mask, d.reduce_axis = 7, 1
        for slot in range(3):
            d.reduce_out[slot] = 1 << 12
    cfg = (ctypes.c_int32 * 4)()
    return _abi.load_library().fuseml_gemm_epilogue_ksplit(ctypes.byref(d), cfg), tuple(cfg[:2])


def test_a_round_that_is_begun_is_priced_whole():
    """Measured slower on the K-split kernel (tiled and K-split us): 10.8 and 14.6,
    30.8 and 39.5, 26.1 and 32.5, 51.9 and 76.9, a little more than one or two rounds."""
    for shape in ((182, 2944, 1024), (1808, 416, 4728), (1507, 440, 4272), (1069, 992, 7600)):
        assert _route(*shape)[0] == 0, shape
    # 256 tiles of 32x64 are one round; with 257 or more that tile is left
    assert _route(500, 1023, 2056) == (1, (32, 64)) and _route(500, 1025, 2056)[1] != (32, 64)


def test_row_reductions_are_priced():
    """Their atomics queue where few rows meet many column tiles: 7.8 us tiled, 8.8."""
    assert _route(20, 4096, 192) == (1, (16, 32))
    assert _route(20, 4096, 192, row_reductions=True)[0] == 0
