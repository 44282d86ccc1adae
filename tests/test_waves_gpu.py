"""The product whose waves share out K (csrc/int8_gemm_waves.hip) at the edges of its tiles, steps and alignments,
against the oracle, bit for bit: every tile shape of both layouts of B, depths around one 64-deep step and around the
steps a wave keeps in flight, columns around a tile's end (B stored K x N: the last tile moves back), rows that start on
no dword, slices of K, batches, every signedness and zero-point form; and the three result kinds of its store."""
from __future__ import annotations

import numpy as np
import pytest

import cases
import oracle
import onegpu_hip as og
from gpu_rig import device, run, run_int32, say

pytestmark = pytest.mark.gpu

# (m, n, k, batch): the tile each takes is in the comment; odd sizes put a ragged edge on every side of it.
SHAPES = [(1, 16, 16, 1), (16, 17, 63, 1), (3, 385, 65, 1), (15, 250, 129, 3),       # 16 x 16
          (5, 4099, 80, 1), (2, 515, 191, 12),                                        # 16 x 32
          (1, 8200, 77, 1), (16, 12001, 130, 1),                                      # 16 x 64
          (1, 20001, 96, 1), (4, 2051, 47, 17),                                       # 16 x 128, or one wave
          (2, 200, 8200, 1), (16, 321, 6500, 1), (1, 1537, 4100, 1),                  # slices of a deep K
          (17, 33, 16, 1), (31, 95, 383, 2), (65, 47, 1601, 1), (40, 40, 3600, 1),    # 32 x 32, two and four waves, slices
          (60, 1057, 5121, 1), (70, 500, 5150, 2), (90, 1999, 5153, 1), (100, 1000, 5184, 2),   # 32 x 64, 64 x 64 in slices
          (129, 1100, 321, 1), (33, 2049, 257, 1), (33, 6001, 100, 1),                # 32 x 32 on all CUs, 32 x 64
          (300, 700, 97, 3),                                                          # 64 x 64
          (333, 65, 95, 60), (257, 500, 33, 40), (500, 1025, 650, 2), (30, 2100, 130, 20)]   # more than one round

# The instances that these shapes run off a dword: tile and waves, "-splitk" in slices of K (of a deep K x N alone at 16 rows).
INSTANCES = {"16x16x4", "16x32x4", "16x64x4", "16x64x1", "32x32x2", "32x32x4", "32x32x4-splitk", "32x64x4", "32x64x4-splitk",
             "32x64x1", "64x64x4", "64x64x4-splitk", "64x64x2"}


@pytest.mark.parametrize("trans", [False, True], ids=["K x N", "N x K"])
def test_sums_are_bit_exact(trans):
    d = device()
    gemm = og.Int8Gemm(d)
    bad_total, kernels = 0, set()
    for i, (m, n, k, batch) in enumerate(SHAPES):
        for v in range(2):
            off, extra = (0, 0) if v == 0 else (1 + i % 3, 1 + (i + 1) % 5)   # rows on, and off, a dword
            c = cases.Case(f"waves {m}x{n}x{k} b{batch} off {off}",
                           cases.problem(m, n, k, batch=batch, trans_b=trans, off_a=off, off_b=off, lda_extra=extra,
                                         ldb_extra=extra), (i & 1) != 0, ((i >> 1) & 1) == v, (i + v) % 3, (i // 3 + v) % 3)
            say(f"{c.name} {'N x K' if trans else 'K x N'} signed {c.a_signed}/{c.b_signed} zp {c.za_mode}/{c.zb_mode}")
            bad, kernel = run_int32(d, gemm, c, 500 + i)
            if bad:
                say(f"  {kernel}: {bad} wrong")
            if v == 1:
                kernels.add(kernel)
            bad_total += bad
    assert bad_total == 0
    assert kernels == {"mfma-i8-waves" + i for i in INSTANCES | (set() if trans else {"16x128x4", "16x64x4-splitk"})}


@pytest.mark.parametrize("m, n, k", [(7, 385, 129), (40, 70, 333), (200, 300, 97), (33, 40, 3600), (60, 1057, 5121),
                                     (90, 1999, 5153), (100, 2000, 5184)])
def test_float_ranged_and_requantized_stores(m, n, k):
    # Whole 16-byte pieces of C's rows (n % 4 == 0) and single values, with and without slices.
    d = device()
    gemm = og.Int8Gemm(d)
    rng = np.random.default_rng(m * n + k)
    a, b = rng.integers(0, 256, m * k + 4, dtype=np.uint8), rng.integers(0, 256, n * k + 4, dtype=np.uint8)
    za, ib = np.array([131, 0, 0, 0], np.uint8), rng.integers(-5000, 5000, n).astype(np.int32)
    scale, fb = (rng.random(n) * 1e-4).astype(np.float32), rng.standard_normal(n).astype(np.float32)
    mult = (rng.random(n) * 2e-5).astype(np.float32)
    sums = oracle.int8_gemm(cases.problem(m, n, k), a, False, b, True, (za[:1], False, 0))
    ba, bb, bz = d.CreateBuffer(a), d.CreateBuffer(b.view(np.int8)), d.CreateBuffer(za)
    bs, bf, bi, bm = (d.CreateBuffer(x) for x in (scale, fb, ib, mult))
    act = np.float32(0.37)
    bact = d.CreateBuffer(np.array([act], np.float32))
    bc, y = d.CreateBufferOf(og.ElementType.Float32, m * n), d.CreateBufferOf(og.ElementType.UInt8, (m * n + 3) // 4 * 4)
    ranges = og.Int8Ranges(d.CreateBufferOf(og.ElementType.Float32, 2 * og.OG_RANGES_MAX))
    p, zpa = og.Int8GemmProblem(m, n, k), og.Int8Operand(bz, 0)
    vec = lambda x: og.Int8Operand(x, 0, True)   # noqa: E731
    say(f"waves stores {m}x{n}x{k}: float, ranged")
    run(d, lambda e: gemm.EncodeFloatRanged(e, p, ba, bb, bc, vec(bs), ranges, zpa, None, vec(bf), vec(bi), og.Int8Operand(bact, 0)))
    want = oracle.float_epilogue(sums, n, (act * scale).astype(np.float32), True, ib, fb)
    got = bc.Read()
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    r = ranges.Buffer.Read()[:2 * ranges.Groups].reshape(-1, 2)
    assert r[:, 0].min() == want.min() and r[:, 1].max() == want.max()
    say(f"waves stores {m}x{n}x{k}: requantized")
    run(d, lambda e: gemm.EncodeRequantized(e, p, ba, bb, y, og.Int8Operand(bm, 0, True), 131, zpa, None, vec(bi)))
    assert d.LastKernel.startswith("mfma-i8-waves"), d.LastKernel
    assert np.array_equal(y.Read()[:m * n], oracle.requant_array(sums, n, mult, True, 131, True, ib))


@pytest.mark.parametrize("m, n, k", [(1000, 700, 1030), (777, 901, 1100), (520, 1030, 1024), (2048, 449, 70), (90, 6000, 130),
                                     (300, 2048, 1087)])
def test_a_grid_of_tiles_for_the_xcds(m, n, k):
    # 64 x 64 tiles, B stored K x N: each XCD takes a block of them; the last blocks of a row and column are part empty.
    d = device()
    c = cases.Case(f"waves grid {m}x{n}x{k}", cases.problem(m, n, k), False, True, 2, 1)
    say(c.name)
    bad, kernel = run_int32(d, og.Int8Gemm(d), c, m + n)
    assert bad == 0 and kernel == "mfma-i8-waves64x64x4", (bad, kernel)


def test_a_grid_of_tiles_records_every_range():
    test_float_ranged_and_requantized_stores(777, 900, 1088)
