"""Consecutive draws of a pass that share one launch group, bit for bit
against the oracle: draws with their own uniforms, textures, culling,
interpolation, viewports and instance counts, of sizes around a wave of
primitives, with triangles across the clip planes and over many tiles."""
import numpy as np
import pytest

import wgc
from oracle import bridge
from wgc import runner, scenes

from test_gpu_parity import announce, assert_parity, clip_color_draw, random_clip_triangles

pytestmark = pytest.mark.gpu


def triangles(n, seed, w, h, depth, blend=wgc.BLEND_REPLACE, **kw):
    vb = random_clip_triangles(n, seed, w, h, spread=1.3, size_px=(3.0, 70.0), w_range=(0.5, 2.0),
                               z_levels=[0.3, 0.5, 0.7], alpha=(0.2, 0.8))
    vb[::9, :, 2] = -0.2 * vb[::9, :, 3]          # some beyond the near plane
    vb[4::13, 0, 2] = 1.3 * vb[4::13, 0, 3]
    return clip_color_draw(vb, depth=depth, blend=blend, **kw)


def both(spec, dev):
    assert_parity(spec, dev)
    assert_parity(scenes.as_wgsl(spec), dev)


@pytest.mark.parametrize("mode", [(wgc.LESS, True), (wgc.GREATER_EQUAL, True), (wgc.LESS, False), (wgc.ALWAYS, True),
                                  (wgc.NOT_EQUAL, True), None, "blend"],
                         ids=["less", "greater_equal", "less_no_write", "always", "not_equal", "no_depth", "blend"])
@pytest.mark.parametrize("sizes", [(1, 63, 64, 65, 200), (700, 1, 900)], ids=["around_a_wave", "large"])
def test_draws_of_one_pass(gpu_device, gpu_device_ext, mode, sizes):
    w, h = 171, 133
    ext = mode == "blend"
    depth = None if ext else mode
    draws = [triangles(n, 7000 + 10 * k, w, h, depth, wgc.BLEND_ALPHA if ext else wgc.BLEND_REPLACE)
             for k, n in enumerate(sizes)]
    draws[1].cull_mode = wgc.CULL_BACK
    draws[1].instance_count = 2
    draws[2].viewport = (-20.0, 9.0, 190.0, 140.0, 0.0, 1.0)
    draws[0].interp = wgc.INTERP_FLAT
    spec = scenes.PassSpec(w, h, clear_color=(0.1, 0.2, 0.3, 1.0), has_depth=depth is not None, clear_depth=0.6,
                           draws=draws, semantics=wgc.SEMANTICS_EXTENDED if ext else wgc.SEMANTICS_REFERENCE,
                           name=f"draws of one pass {mode} {sizes}")
    both(spec, gpu_device_ext if ext else gpu_device)


def test_groups_break_where_the_rule_changes(gpu_device_ext):
    """Opaque, blended and opaque draws, one with a scissor rect of its own."""
    w, h = 130, 90
    draws = [triangles(150, 7100, w, h, (wgc.LESS, True)), triangles(90, 7101, w, h, (wgc.LESS, True)),
             triangles(120, 7102, w, h, (wgc.LESS, False), wgc.BLEND_ALPHA),
             triangles(80, 7103, w, h, (wgc.LESS, False), wgc.BLEND_ALPHA),
             triangles(110, 7104, w, h, (wgc.LESS, True)), triangles(60, 7105, w, h, (wgc.LESS, True))]
    draws[4].scissor = (20, 10, 77, 61)
    spec = scenes.PassSpec(w, h, has_depth=True, clear_depth=1.0, draws=draws, semantics=wgc.SEMANTICS_EXTENDED,
                           name="groups of draws")
    both(spec, gpu_device_ext)


@pytest.mark.parametrize("tile", [0, 1, 6])
def test_textured_objects_with_their_own_uniforms(gpu_device, tile):
    w, h = 200, 150
    draws = []
    for k in range(5):
        d = scenes.config2_textured(seed=50 + k, width=w, height=h, segments=12, rings=6 + k).draws[0]
        size = 8 << k
        d.texture = (size, size, scenes.checker_texture(size, 3, 16, 90 + k), k % 2 == 1)
        d.uniform = scenes.perspective_view(45.0 + 12 * k, w / h, 0.1, 10.0, 2.0 + 0.4 * k)
        d.address_u = (wgc.REPEAT, wgc.CLAMP_TO_EDGE, wgc.MIRROR_REPEAT)[k % 3]
        draws.append(d)
    spec = scenes.PassSpec(w, h, has_depth=True, clear_depth=1.0, draws=draws, name=f"objects, tile option {tile}")
    gpu_device.set_option(wgc.OPTION_RASTER_TILE, tile)
    try:
        both(spec, gpu_device)
    finally:
        gpu_device.set_option(wgc.OPTION_RASTER_TILE, 0)


def test_primitive_index_and_big_triangles_across_draws(gpu_device):
    """@builtin(primitive_index) counts from each draw's first primitive; a
    triangle over the whole target in each draw goes through the big list."""
    w, h = 260, 180
    draws = []
    for k in range(3):
        d = scenes.fragment_test_scene(scenes.FS_PRIM_RED, scenes.EARLY_NONE, n=100 + 33 * k, width=w, height=h,
                                       seed=7200 + k).draws[0]
        vb = np.frombuffer(d.vertex_data, np.float32).copy().reshape(-1, 3, 8)
        vb[7, :, :2] = ((-3.0, -3.0), (3.0, -3.0), (0.0, 4.0))
        d.vertex_data = vb.tobytes()
        draws.append(d)
    spec = scenes.PassSpec(w, h, clear_color=(0, 0, 0, 1), has_depth=True, clear_depth=0.7, draws=draws,
                           name="primitive index across draws")
    assert_parity(spec, gpu_device)


def test_noalloc_draws_one_at_a_time_equals_the_group(gpu_device):
    announce("draws of one pass, allocation-free")
    w, h = 171, 133
    draws = [triangles(n, 7300 + n, w, h, (wgc.LESS, True)) for n in (40, 300, 65)]
    spec = scenes.PassSpec(w, h, has_depth=True, clear_depth=1.0, draws=draws)
    pp = runner.PreparedPass(gpu_device, spec)
    pp.submit()
    want = pp.result()
    rng = np.random.default_rng(7)
    gpu_device.write_texture(pp.res[0].color, rng.integers(0, 256, w * h * 4, dtype=np.uint8).tobytes())
    gpu_device.write_texture(pp.res[0].depth, rng.random(w * h, dtype=np.float32).tobytes())
    gpu_device.submit_noalloc([pp.command_buffer])
    got = pp.result()
    ref = bridge.render(spec)
    for r in (want, got):
        assert r.fragments == ref.fragments
        assert np.array_equal(r.color, ref.color)
        assert np.array_equal(r.depth.view(np.uint32), ref.depth.view(np.uint32))


@pytest.mark.parametrize("blend", [False, True])
def test_each_draw_keeps_its_clip_slots(gpu_device_ext, blend):
    """Small draws whose triangles cross most of the clip planes: each has
    more sub-triangles than two per primitive (about ten), which a draw of
    few primitives has slots for, and so have the draws of a pass together."""
    w, h, n = 150, 110, 60
    draws, subs = [], 0
    for k in range(12):
        u = scenes.splitmix_f32(7400 + k, n * 8).reshape(n, 8)
        vb = np.zeros((n, 3, 8), np.float32)
        ang = 2.0 * np.pi * (u[:, :1] + np.arange(3) / 3.0)
        vb[:, :, 0], vb[:, :, 1] = 2.2 * np.cos(ang), 2.2 * np.sin(ang)
        vb[:, :, 2] = np.where(u[:, 1:2] < 0.5, (-0.4, 0.5, 1.5), (1.4, -0.3, 0.6))
        vb[:, :, 3] = 1.0
        vb[:, :, 4:8] = u[:, None, 4:8]
        of_draw = sum(len(bridge.clip_triangle(t[:, :4])) for t in vb)
        assert 2 * n < of_draw <= 2 * n + 1024
        subs += of_draw
        draws.append(clip_color_draw(vb, depth=None if blend else (wgc.LESS, True),
                                     blend=wgc.BLEND_ALPHA if blend else wgc.BLEND_REPLACE))
    assert subs > 2 * 64 * len(draws) + 1024
    spec = scenes.PassSpec(w, h, has_depth=not blend, clear_depth=1.0, draws=draws, semantics=wgc.SEMANTICS_EXTENDED,
                           name=f"clip slots of merged draws blend={blend}")
    both(spec, gpu_device_ext)


def test_batching_off_is_one_launch_set_per_draw(gpu_device):
    announce("draws of one pass, batching off")
    w, h = 171, 133
    draws = [triangles(n, 7500 + n, w, h, (wgc.LESS, True)) for n in (40, 300, 65)]
    spec = scenes.PassSpec(w, h, has_depth=True, clear_depth=1.0, draws=draws)

    def launches(spec):
        got = runner.render(spec, gpu_device)
        assert np.array_equal(got.color, bridge.render(spec).color)
        return gpu_device.last_pass_stats().kernel_launches

    merged = launches(spec)
    gpu_device.set_option(wgc.OPTION_BATCHING, 0)
    try:
        alone = [launches(scenes.PassSpec(w, h, has_depth=True, clear_depth=1.0, draws=[d])) for d in draws]
        assert launches(spec) == sum(alone) > merged
    finally:
        gpu_device.set_option(wgc.OPTION_BATCHING, 1)


# Groups too large for setup to clip in place (a launch for the clipper, no
# clear ahead of the tiles), with tiles of several batches that stay whole,
# and one of more primitives than a group takes.
@pytest.mark.parametrize("mode,count,n,launches", [("less", 5, 60000, 3), ("no_depth", 5, 60000, 3),
                                                   ("blend", 5, 60000, 3), ("less", 9, 125000, 5)],
                         ids=["less", "no_depth", "blend", "two_groups"])
def test_large_groups(gpu_device_ext, mode, count, n, launches):
    w, h = 1600, 900
    depth, blend = (wgc.LESS, True) if mode == "less" else None, wgc.BLEND_ALPHA if mode == "blend" else wgc.BLEND_REPLACE
    draws = []
    for k in range(count):
        vb = random_clip_triangles(n, 7600 + k, w, h, spread=1.03, size_px=(1.0, 14.0 if count < 9 else 5.0),
                                   w_range=(0.5, 2.0), z_levels=[0.3, 0.5, 0.7], alpha=(0.2, 0.8))
        vb[::9, :, 2] = -0.2 * vb[::9, :, 3]
        vb[4::13, 0, 2] = 1.3 * vb[4::13, 0, 3]
        draws.append(clip_color_draw(vb, depth=depth, blend=blend))
    draws[1].cull_mode = wgc.CULL_BACK
    draws[2].viewport = (-20.0, 9.0, 1700.0, 870.0, 0.0, 1.0)
    spec = scenes.PassSpec(w, h, clear_color=(0.1, 0.2, 0.3, 1.0), has_depth=depth is not None, clear_depth=1.0,
                           draws=draws, semantics=wgc.SEMANTICS_EXTENDED, name=f"large groups {mode} {count} x {n}")
    assert_parity(spec, gpu_device_ext)
    assert gpu_device_ext.last_pass_stats().kernel_launches == launches
    if count < 9:
        assert_parity(scenes.as_wgsl(spec), gpu_device_ext)
