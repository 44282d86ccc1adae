"""Int8GemmOptions.Tile keeps the kernel it names, whatever the size (include/onegpu_hip.h, OG_GEMM_NO_SKINNY and the flags
after it): the kernels that the product's launches run, both of a split product's, and its sums."""
from __future__ import annotations

import numpy as np
import pytest

import cases
import oracle
import onegpu_hip as og
from gpu_rig import device, say, to_problem
from test_quant_gpu import run_named

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile, m, n, k, want", [
    (32, 5, 1000, 2000, ["mfma-i8-rows16-splitk", "skinny-reduce"]),      # rows off 16 bytes
    (32, 16, 2048, 2048, ["mfma-i8-rows16-splitk", "skinny-reduce"]),
    (64, 4, 1024, 2048, ["mfma-i8-direct128x128x64-splitk", "splitk-sum"]),
    (64, 256, 256, 2304, ["mfma-i8-direct128x128x64-splitk", "splitk-sum"])])
def test_a_pinned_kernel_runs(tile, m, n, k, want):
    d = device()
    gemm = og.Int8Gemm(d, og.Int8GemmOptions(Tile=tile))
    rng = np.random.default_rng(m + n + k)
    a, b = rng.integers(0, 256, m * k, dtype=np.uint8), rng.integers(0, 256, k * n, dtype=np.uint8)
    p = cases.problem(m, n, k)
    ba, bb = d.CreateBuffer(a), d.CreateBuffer(b.view(np.int8))
    c = d.CreateBufferOf(og.ElementType.Int32, m * n)
    say(f"pinned {tile}: {m}x{n}x{k}")
    names = run_named(d, lambda e: gemm.EncodeInt32(e, to_problem(p), ba, bb, c))
    assert names == want
    assert np.array_equal(c.Read(), oracle.int8_gemm(p, a, False, b, True))
