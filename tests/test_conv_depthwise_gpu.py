"""Depthwise ConvInteger by tiles (csrc/conv.hip, k_conv_depthwise_tile) at the edges of what it takes: images smaller than a
quad of columns or the window, rows and columns that end inside a quad or a group of rows, several row or column tiles,
several planes a tile, strides, one-sided and over-wide padding, several output channels an input channel, one dimension;
windows just outside it, and convolutions on either side of the sizes it is chosen for, beside them; against the oracle,
bit for bit."""
from __future__ import annotations

import pytest

import cases
from gpu_rig import device, say
from test_conv_gpu import _configs, _run_case

pytestmark = pytest.mark.gpu

# (batch, cin, h, w, multiplier, kh, kw, strides (h, w), pads (top, left, bottom, right), dilation, by tiles)
GEOMETRIES = [
    (1, 3, 2, 3, 1, 5, 5, (1, 1), (3, 2, 3, 2), 1, True),         # 4 x 3 outputs
    (45, 256, 4, 4, 1, 3, 3, (1, 1), (1, 1, 1, 1), 1, True),      # one quad, one group of rows
    (29, 128, 5, 5, 2, 3, 3, (1, 1), (1, 1, 1, 1), 1, True),      # one past both
    (3, 7, 9, 13, 3, 5, 5, (1, 1), (2, 2, 2, 2), 1, True),
    (63, 50, 31, 32, 1, 3, 3, (2, 2), (1, 1, 1, 1), 1, True),     # 16 x 16 outputs
    (2, 6, 17, 19, 1, 5, 5, (2, 2), (2, 2, 2, 2), 1, True),
    (45, 185, 20, 21, 1, 3, 3, (2, 2), (0, 1, 1, 0), 1, True),
    (1, 5, 11, 6, 1, 5, 5, (1, 1), (7, 0, 0, 9), 1, True),        # whole rows and columns of padding
    (2, 16, 70, 90, 1, 3, 3, (1, 1), (0, 0, 0, 0), 1, True),      # several row tiles
    (2, 14, 6, 1100, 1, 3, 3, (1, 1), (1, 1, 1, 1), 1, True),     # two column tiles
    (1, 1, 7, 2200, 1, 5, 5, (2, 2), (2, 2, 2, 2), 1, True),
    (14, 300, 7, 7, 1, 3, 3, (1, 1), (1, 1, 1, 1), 1, True),      # sixteen planes a tile
    (2, 300, 7, 7, 1, 5, 5, (1, 1), (2, 2, 2, 2), 1, True),       # two
    (5, 205, 3, 3, 1, 5, 5, (2, 2), (2, 2, 2, 2), 1, True),       # four, the last tile of fewer
    (2, 130, 1, 333, 1, 1, 3, (1, 1), (0, 1, 0, 1), 1, True),     # one dimension
    (2, 109, 1, 1500, 1, 1, 5, (2, 2), (0, 2, 0, 2), 1, True),
    (2, 800, 1, 101, 2, 1, 3, (1, 2), (0, 0, 0, 0), 1, True),
    (5, 65, 9, 30, 1, 1, 5, (1, 1), (1, 2, 2, 2), 1, True),       # a row window over an image
    (20, 100, 9, 31, 1, 1, 3, (2, 2), (0, 1, 0, 1), 1, True),
    (600, 70, 1, 2, 1, 1, 3, (1, 1), (0, 1, 0, 1), 1, True),
    (1, 1, 1, 1, 1, 3, 3, (1, 1), (1, 1, 1, 1), 1, False),        # too few outputs, or on too small planes
    (2, 5, 4, 4, 1, 3, 3, (1, 1), (1, 1, 1, 1), 1, False),
    (50, 500, 3, 3, 1, 3, 3, (1, 1), (1, 1, 1, 1), 1, False),
    (4, 205, 20, 21, 1, 3, 3, (2, 2), (0, 1, 1, 0), 1, False),
    (7, 600, 3, 3, 1, 5, 5, (2, 2), (2, 2, 2, 2), 1, False),
    (1, 33, 1, 333, 1, 1, 3, (1, 1), (0, 1, 0, 1), 1, False),
    (1, 4, 120, 131, 4, 3, 3, (1, 1), (2, 2, 2, 2), 2, False),    # not tiled: dilated, unequal strides, other windows
    (1, 4, 120, 131, 8, 3, 3, (1, 2), (1, 1, 1, 1), 1, False),
    (1, 4, 220, 231, 9, 3, 3, (3, 3), (1, 1, 1, 1), 1, False),
    (1, 4, 12, 13, 1, 5, 3, (1, 1), (2, 1, 2, 1), 1, False),
    (1, 4, 12, 13, 1, 7, 7, (1, 1), (3, 3, 3, 3), 1, False)]


@pytest.mark.parametrize("index", range(len(GEOMETRIES)))
def test_depthwise_tiles_are_bit_exact(index):
    b, ci, h, w, mult, kh, kw, strides, pads, dil, tiles = GEOMETRIES[index]
    d = device()
    conv = _configs(d)[0][1]
    p = cases.conv_problem(b, ci, h, w, ci * mult, kh, kw, groups=ci, dilation=dil)
    p.update(StrideHeight=strides[0], StrideWidth=strides[1], PadTop=pads[0], PadLeft=pads[1], PadBottom=pads[2],
             PadRight=pads[3])
    for s in range(4):
        c = dict(name=f"depthwise {b}x{ci}x{h}x{w} x {mult}, {kh}x{kw}", p=p, xs=(s & 1) != 0, ws=(s & 2) != 0,
                 xzm=(index + s) % 2, wzm=(index + s // 2) % 3, fill=-1, scratch_images=0)
        say(f"{c['name']} strides {strides} pads {pads} dilation {dil} signed {c['xs']}/{c['ws']} zp {c['xzm']}/{c['wzm']}")
        bad, kern = _run_case(d, conv, c, 9000 + 10 * index + s)
        assert kern == ("conv-depthwise-tile-i8" if tiles else "conv-depthwise-i8")
        assert bad == 0, f"{c['name']}: {bad} elements differ"
