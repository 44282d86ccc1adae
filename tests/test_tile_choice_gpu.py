"""Products of the 256 x 256 class whose padding, or whose byte sums over partial tiles, send them to the 128 tile
(direct_uses_large, csrc/int8_gemm_direct.hip), on both sides of its line, against the oracle, bit for bit; the ranged
form too, whose pairs then come from the 128 tile's epilogue."""
from __future__ import annotations

import numpy as np
import pytest

import cases
import oracle
import onegpu_hip as og
from gpu_rig import device, run, run_int32, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m, n, k, batch, trans, za, zb, b_signed, tile", [
    (40, 304, 64, 200, False, 1, 0, True, 128), (129, 272, 128, 104, True, 2, 2, True, 128),     # padding; byte sums
    (256, 256, 64, 200, True, 1, 1, False, 256), (250, 512, 64, 101, False, 1, 0, True, 256),     # whole; little padding
    (130, 256, 2048, 200, False, 0, 0, True, 256), (250, 256, 2048, 200, True, 1, 2, True, 256),  # a deep K
    (120, 256, 2048, 200, False, 0, 0, True, 128)])
def test_sums_are_bit_exact(m, n, k, batch, trans, za, zb, b_signed, tile):
    d = device()
    c = cases.Case(f"tile choice {m}x{n}x{k} b{batch}", cases.problem(m, n, k, batch=batch, trans_b=trans, share_b=True),
                   False, b_signed, za, zb)
    say(c.name)
    bad, kernel = run_int32(d, og.Int8Gemm(d), c, m + n)
    assert bad == 0 and kernel == f"mfma-i8-direct{tile}x{tile}x64", (bad, kernel)


def test_ranged_product_of_the_class():
    d = device()
    m, n, k, batch = 40, 304, 64, 200
    rng = np.random.default_rng(5)
    a, b = rng.integers(0, 256, batch * m * k, dtype=np.uint8), rng.integers(0, 256, batch * n * k, dtype=np.uint8)
    scale = (rng.random(n) * 1e-3).astype(np.float32)
    p = oracle.Gemm(m, n, k, Batch=batch, StrideA=m * k, StrideB=n * k)
    want = oracle.float_epilogue(oracle.int8_gemm(p, a, False, b, True), n, scale, True)
    q = og.Int8GemmProblem(m, n, k)
    q.Batch, q.StrideA, q.StrideB = batch, m * k, n * k
    bc = d.CreateBufferOf(og.ElementType.Float32, batch * m * n)
    ranges = og.Int8Ranges(d.CreateBufferOf(og.ElementType.Float32, 2 * og.OG_RANGES_MAX))
    say("tile choice: ranged product")
    run(d, lambda e: og.Int8Gemm(d).EncodeFloatRanged(e, q, d.CreateBuffer(a), d.CreateBuffer(b.view(np.int8)), bc,
                                                      og.Int8Operand(d.CreateBuffer(scale), 0, True), ranges))
    assert d.LastKernel == "mfma-i8-direct128x128x64", d.LastKernel
    assert np.array_equal(bc.Read().view(np.uint32), want.view(np.uint32))
    r = ranges.Buffer.Read()[:2 * ranges.Groups].reshape(-1, 2)
    assert r[:, 0].min() == want.min() and r[:, 1].max() == want.max()
