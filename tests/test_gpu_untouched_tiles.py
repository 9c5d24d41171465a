"""Tiles that only the clear or a draw's big triangles reach, bit for bit
against the oracle: targets of odd and aligned widths, one and many passes,
more tiles than one look-up of a workgroup holds, every tile shape."""
import numpy as np
import pytest

import wgc
from oracle import bridge
from wgc import runner, scenes

from test_gpu_parity import announce, assert_parity, clip_color_draw, random_clip_triangles

pytestmark = pytest.mark.gpu

SIZES = [(516, 260), (333, 97), (64, 64), (67, 33), (4, 4), (1, 130), (1028, 37), (260, 515)]


def spec(i, w, h, ordered, clear):
    vb = random_clip_triangles(3 + i % 3, 8400 + i, w, h, spread=0.6, size_px=(0.2 * max(w, h), 0.9 * max(w, h)),
                               z_levels=[0.2, 0.4, 0.6], alpha=(0.3, 0.8))
    small = random_clip_triangles(40, 8500 + i, w, h, spread=0.2, size_px=(2.0, 9.0), z_levels=[0.3, 0.5],
                                  alpha=(0.3, 0.8))
    draw = clip_color_draw(np.concatenate([vb, small]) if i % 2 else vb, depth=(wgc.LESS, True),
                           blend=wgc.BLEND_ALPHA if ordered else wgc.BLEND_REPLACE)
    s = scenes.PassSpec(w, h, clear_color=(0.2, 0.4, 0.6, 0.8) if clear != "depth" else None, has_depth=True,
                        clear_depth=0.55 if clear != "color" else None, draws=[draw],
                        semantics=wgc.SEMANTICS_EXTENDED, name=f"untouched {w}x{h} {ordered} {clear}")
    rng = np.random.default_rng(i)
    s.color_init = rng.integers(0, 256, (h, w, 4), dtype=np.uint8).tobytes()
    s.depth_init = rng.random((h, w), dtype=np.float32).tobytes()
    return s


@pytest.mark.parametrize("ordered", [False, True], ids=["opaque", "blended"])
@pytest.mark.parametrize("clear", ["both", "color", "depth"])
def test_one_pass_and_a_batch(gpu_device_ext, ordered, clear):
    specs = [spec(i, w, h, ordered, clear) for i, (w, h) in enumerate(SIZES)]
    for s in specs[:3]:
        assert_parity(s, gpu_device_ext)
    announce(f"untouched tiles of a batch {ordered} {clear}")
    for got, s in zip(runner.render_batch(specs, wgc.Device(0, wgc.SEMANTICS_EXTENDED))[0], specs):
        ref = bridge.render(s)
        np.testing.assert_array_equal(got.color, ref.color)
        np.testing.assert_array_equal(got.depth.view(np.uint32), ref.depth.view(np.uint32))


@pytest.mark.parametrize("tile", range(1, 8))
def test_tile_shapes(tile):
    announce(f"untouched tiles, tile option {tile}")
    dev = wgc.Device(0, wgc.SEMANTICS_EXTENDED)
    dev.set_option(wgc.OPTION_RASTER_TILE, tile)
    specs = [spec(i, w, h, False, "both") for i, (w, h) in enumerate(SIZES)]
    for got, s in zip(runner.render_batch(specs, dev)[0], specs):
        ref = bridge.render(s)
        np.testing.assert_array_equal(got.color, ref.color)
        np.testing.assert_array_equal(got.depth.view(np.uint32), ref.depth.view(np.uint32))
