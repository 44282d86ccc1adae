"""ConvInteger without its column matrix (csrc/int8_gemm_waves.hip, CONV): windows read tap by tap where the output is as
wide as the image, and 1 x 1 windows over image rows of any length, at the edges of what they take: planes barely larger
than a tile, windows wider than half the image, dilation, padding on one side, more or fewer output rows than input
ones, depths around one step, groups, batches, slices of K, more tiles than CUs; against the oracle, bit for bit."""
from __future__ import annotations

import pytest

import cases
from gpu_rig import device, say
from test_conv_gpu import _configs, _run_case

pytestmark = pytest.mark.gpu

# (batch, cin, h, w, cout, kh, kw, pads (top, left, bottom, right), dilation (h, w), groups)
GEOMETRIES = [
    (1, 2, 4, 4, 3, 3, 3, (1, 1, 1, 1), (1, 1), 1),          # K = 18, 16 positions: the smallest taken
    (2, 5, 7, 7, 40, 3, 3, (1, 1, 1, 1), (1, 1), 1),         # 49 positions; K = 45
    (1, 64, 14, 14, 33, 3, 3, (1, 1, 1, 1), (1, 1), 1),      # K = 576, whole steps
    (3, 9, 5, 9, 20, 5, 5, (2, 2, 2, 2), (1, 1), 1),         # windows over half the image
    (1, 7, 6, 40, 18, 3, 5, (0, 2, 0, 2), (1, 1), 1),        # fewer output rows than input rows
    (1, 7, 6, 40, 18, 3, 3, (4, 2, 3, 0), (1, 1), 1),        # more of them; columns padded on one side
    (2, 11, 16, 16, 24, 3, 3, (2, 2, 2, 2), (2, 2), 1),      # dilation
    (1, 6, 12, 33, 50, 4, 2, (1, 0, 2, 1), (1, 1), 1),       # even windows
    (1, 80, 1, 333, 70, 1, 3, (0, 1, 0, 1), (1, 1), 1),      # one dimension
    (4, 40, 31, 31, 34, 3, 3, (1, 1, 1, 1), (1, 1), 2),      # groups
    (1, 40, 10, 10, 5, 7, 7, (3, 3, 3, 3), (1, 1), 1),       # 49 taps, few rows
    (1, 600, 8, 8, 40, 3, 3, (1, 1, 1, 1), (1, 1), 1),       # slices of K (5400)
    (8, 10, 50, 50, 96, 3, 3, (1, 1, 1, 1), (1, 1), 1),      # more tiles than CUs
    (4, 37, 7, 9, 65, 1, 1, (0, 0, 0, 0), (1, 1), 1),        # 1 x 1 over rows of 63 bytes
    (30, 20, 31, 31, 100, 1, 1, (0, 0, 0, 0), (1, 1), 1),    # 1 x 1, more tiles than CUs
    (2, 12, 9, 10, 16, 3, 3, (1, 1, 1, 1), (1, 1), 2),       # packed: two groups of a small matrix, many groups, a long
    (1, 48, 14, 14, 96, 3, 3, (1, 1, 1, 1), (1, 1), 12),     # walk on two waves
    (1, 512, 14, 14, 512, 3, 3, (1, 1, 1, 1), (1, 1), 1)]
PACKED = GEOMETRIES[-3:]


@pytest.mark.parametrize("index", range(len(GEOMETRIES)))
def test_convolutions_without_a_column_matrix_are_bit_exact(index):
    b, ci, h, w, co, kh, kw, pads, dil, groups = GEOMETRIES[index]
    d = device()
    conv = _configs(d)[0][1]
    p = cases.conv_problem(b, ci, h, w, co, kh, kw, groups=groups)
    p.update(PadTop=pads[0], PadLeft=pads[1], PadBottom=pads[2], PadRight=pads[3], DilationHeight=dil[0],
             DilationWidth=dil[1])
    for s in range(4):
        c = dict(name=f"conv waves {b}x{ci}x{h}x{w} -> {co}, {kh}x{kw}", p=p, xs=(s & 1) != 0, ws=(s & 2) != 0,
                 xzm=(index + s) % 2, wzm=(index + s) % 3, fill=-1, scratch_images=0)
        say(f"{c['name']} pads {pads} dilation {dil} groups {groups} signed {c['xs']}/{c['ws']} zp {c['xzm']}/{c['wzm']}")
        bad, kern = _run_case(d, conv, c, 7000 + 10 * index + s)
        assert bad == 0, f"{c['name']}: {bad} elements differ ({kern})"
        assert kern.startswith("conv-waves") == (kh * kw > 1 and GEOMETRIES[index] not in PACKED), kern
