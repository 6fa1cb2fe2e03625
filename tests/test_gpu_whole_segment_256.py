"""Whole segments at head size 256 (tiles of 32 tokens, four wavefronts): borders of tiles, blocks of half a tile and more, both sides
of the lines from which the segments are cut into ranges, as in test_gpu_whole_segment.py, whose oracles and tolerances these are."""

import pytest

import test_gpu_whole_segment as W

pytestmark = pytest.mark.gpu
_pkg = W._pkg

CASES = [
    # Hq, Hkv, D, bs, contexts, bfp8, window, sink, forced
    (16, 8, 256, 32, [0, 31, 32, 63, 64, 127], False, 0, False, False),           # up to a tile per wavefront
    (16, 8, 256, 16, [0, 15, 16, 100], False, 0, True, False),                    # tiles of two blocks
    (8, 8, 256, 32, [5, 95, 96, 2000], False, 100, False, False),                 # one head per group, in a window
    (32, 2, 256, 64, [126, 127, 128], False, 0, True, False),                     # sixteen heads; a table of more than 128 tokens: ranges
    (10, 2, 256, 64, [255, 256, 257, 1000], False, 0, False, True),               # as many rounds of tiles as asked for
    (16, 8, 256, 32, [(37 * i) % 256 for i in range(16)], False, 0, True, False),  # half of the CUs: two tiles per wavefront
    (16, 8, 256, 64, [(53 * i) % 256 for i in range(33)], False, 0, False, False),  # more segments than CUs: ranges
    (16, 8, 256, 32, [0, 31, 32, 127], True, 0, False, False),                    # block-float-8
    (6, 3, 256, 48, [40, 333, 700], True, 90, True, False),
    (16, 8, 256, 64, [(29 * i) % 256 for i in range(20)], True, 0, False, False),
]


@pytest.mark.parametrize("hq,hkv,d,bs,ctx,bfp8,window,with_sink,forced", CASES)
def test_whole_segments_equal_ranges(monkeypatch, hq, hkv, d, bs, ctx, bfp8, window, with_sink, forced):
    W.test_whole_segments_equal_ranges(monkeypatch, hq, hkv, d, bs, ctx, bfp8, window, with_sink, forced)


@pytest.mark.parametrize("bfp8", [False, True])
def test_rows_of_odd_strides_and_parked_users(bfp8):
    W.test_whole_segments_with_rows_of_odd_strides_and_parked_users(256, bfp8)
