"""Scratch that is refused: merged draws fall back to smaller groups, passes
to the first lane, and the second lane's arena makes room, with the pictures
of the oracle throughout."""
import numpy as np
import pytest

import wgc
from oracle import bridge
from wgc import runner, scenes

from test_gpu_parity import announce, clip_color_draw, random_clip_triangles
from test_gpu_topology import crowded_lines

pytestmark = pytest.mark.gpu

MIB = 1 << 20


def one_draw(n, seed, w, h, blend=True):
    vb = random_clip_triangles(n, seed, w, h, size_px=(2.0, 12.0), alpha=(0.2, 0.8))
    return clip_color_draw(vb, depth=None if blend else (wgc.LESS, True),
                           blend=wgc.BLEND_ALPHA if blend else wgc.BLEND_REPLACE)


def spec_of(draws, w, h, blend=True, name=""):
    return scenes.PassSpec(w, h, clear_color=(0.1, 0.2, 0.3, 1.0), has_depth=not blend, clear_depth=1.0, draws=draws,
                           semantics=wgc.SEMANTICS_EXTENDED, name=name)


def check(passes, refs):
    for p, ref in zip(passes, refs):
        got = p.results()[0]
        np.testing.assert_array_equal(got.color, ref.color)
        if ref.depth is not None:
            np.testing.assert_array_equal(got.depth.view(np.uint32), ref.depth.view(np.uint32))


@pytest.mark.parametrize("blend", [False, True])
def test_merged_draws_without_room(blend):
    """Six draws of 40000 triangles are one group, in less memory fewer, and
    where only one draw's scratch (about 1.1 KB a triangle) fits they run one
    after another; with less than that the submission is refused."""
    announce(f"merged draws without room, blend={blend}")
    w, h = 300, 200
    dev = wgc.Device(0, wgc.SEMANTICS_EXTENDED)
    spec = spec_of([one_draw(40000, 9000 + k, w, h, blend) for k in range(6)], w, h, blend)
    ref = bridge.render(spec)
    p = runner.PreparedPass(dev, spec)
    launches = []
    for mib in (0, 200, 75):
        dev.debug_scratch_limit(mib * MIB)
        p.submit()
        check([p], [ref])
        launches.append(dev.last_pass_stats().kernel_launches)
    assert launches[0] < launches[1] < launches[2], launches
    dev.debug_scratch_limit(20 * MIB)
    with pytest.raises(wgc.WgcError) as e:
        p.submit()
    assert e.value.code == wgc.ERR_OUT_OF_MEMORY
    dev.debug_scratch_limit()
    p.submit()
    check([p], [ref])


@pytest.mark.parametrize("mib", [0, 100])
def test_lane_without_an_arena(mib):
    """Independent passes in turn where the second lane gets an arena and
    where it does not (64 MiB at least each)."""
    announce(f"lane without an arena, {mib} MiB")
    dev = wgc.Device(0, wgc.SEMANTICS_EXTENDED)
    dev.debug_scratch_limit(mib * MIB)
    specs = [spec_of([one_draw(3000 + 500 * k, 9100 + k, 120 + k, 90)], 120 + k, 90) for k in range(3)]
    refs = [bridge.render(s) for s in specs]
    passes = [runner.PreparedPass(dev, s) for s in specs]
    for _ in range(8):
        for p in passes:
            p.submit()
    check(passes, refs)


@pytest.mark.parametrize("mib", [0, 200])
def test_arenas_that_grow_under_older_plans(mib):
    """Small passes on both lanes, then passes of more scratch, then the small
    ones again.  Of 200 MiB both lanes' first arenas take 64 each, and the
    first lane's larger one only fits once the second has given way."""
    announce(f"arenas that grow, {mib} MiB")
    dev = wgc.Device(0, wgc.SEMANTICS_EXTENDED)
    dev.debug_scratch_limit(mib * MIB)
    sizes = [(3000, 120), (2000, 130), (110000, 140), (100000, 150), (900, 160)]
    specs = [spec_of([one_draw(n, 9200 + n, w, 90)], w, 90) for n, w in sizes]
    refs = [bridge.render(s) for s in specs]
    passes = [runner.PreparedPass(dev, s) for s in specs]
    for order in ((0, 1, 4), (0, 1, 4), (2, 3), (0, 1, 4, 2, 3), (4, 3, 1, 0)):
        for _ in range(3):
            for k in order:
                passes[k].submit()
        check([passes[k] for k in order], [refs[k] for k in order])


def test_failed_submissions_beside_running_ones():
    """A pass that is refused when it is submitted (a vertex buffer is not
    bound) among passes on both lanes: the others are whole."""
    announce("failed submissions beside running ones")
    dev = wgc.Device(0, wgc.SEMANTICS_EXTENDED)
    specs = [spec_of([one_draw(6000, 9300 + k, 200 + k, 150)], 200 + k, 150) for k in range(3)]
    refs = [bridge.render(s) for s in specs]
    passes = [runner.PreparedPass(dev, s) for s in specs]
    target = dev.create_texture(64, 64, wgc.RGBA8_UNORM)
    module = dev.create_shader_module_builtin(wgc.PROGRAM_CLIP_COLOR)
    pipeline = dev.create_render_pipeline(module, [(32, wgc.STEP_VERTEX, [(wgc.FLOAT32X4, 0, 0),
                                                                         (wgc.FLOAT32X4, 16, 1)])])
    enc = dev.create_command_encoder()
    rp = enc.begin_render_pass(color=target, clear_color=(0, 0, 0, 1))
    rp.set_pipeline(pipeline)
    rp.draw(range(0, 3))
    rp.end()
    bad = enc.finish()
    for n in range(12):
        for p in passes[:1 + n % 3]:
            p.submit()
        with pytest.raises(wgc.WgcError):
            dev.submit([bad])
    for p in passes:
        p.submit()
    check(passes, refs)
    fragments = sum(r.fragments for r in refs)
    before = dev.totals()[0]
    for p in passes:
        p.submit()
    dev.poll()
    assert dev.totals()[0] - before == fragments


@pytest.mark.parametrize("wgsl", [False, True])
@pytest.mark.parametrize("mode", ["less", "last", "blend"])
def test_lines_without_room(mode, wgsl):
    """Crowded lines with their winners in global memory (2 MiB for this
    target), without (tile bins, 1 MiB), and with records alone (0.12 MiB),
    from an arena (64 MiB at least) and from the static scratch."""
    announce(f"lines without room, {mode} wgsl={wgsl}")
    dev = wgc.Device(0, wgc.SEMANTICS_EXTENDED)
    spec = crowded_lines(1300, 512, 512, mode)
    ref = bridge.render(spec)
    p = runner.PreparedPass(dev, scenes.as_wgsl(spec) if wgsl else spec)
    rng = np.random.default_rng(3)
    for arena, static in ((0, 0), (65 * MIB, 1500 << 10), (64 * MIB + 2048, 200 << 10)):
        dev.debug_scratch_limit(arena, static)
        for submit in (p.submit, lambda: dev.submit_noalloc([p.command_buffer])):
            dev.write_texture(p.res[0].color, rng.integers(0, 256, 512 * 512 * 4, dtype=np.uint8).tobytes())
            submit()
            check([p], [ref])
    dev.debug_scratch_limit(0, 100 << 10)
    with pytest.raises(wgc.WgcError) as e:
        dev.submit_noalloc([p.command_buffer])
    assert e.value.code == wgc.ERR_OUT_OF_MEMORY
