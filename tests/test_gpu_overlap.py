"""Submissions of single passes that may run beside each other: whatever they
share, each sees the results of those submitted before it.  The same passes
with a wait after each submission are the reference here (and the oracle, for
the independent ones)."""
import threading
from types import SimpleNamespace

import numpy as np
import pytest

import wgc
from oracle import bridge
from wgc import runner, scenes

from test_gpu_parity import announce, clip_color_draw, random_clip_triangles

pytestmark = pytest.mark.gpu

SIZE = 96


def blended(n, seed, w=SIZE, h=SIZE, size_px=(5.0, 60.0)):
    vb = random_clip_triangles(n, seed, w, h, size_px=size_px, alpha=(0.2, 0.8))
    return clip_color_draw(vb, depth=None, blend=wgc.BLEND_ALPHA)


def textured(source, k):
    d = scenes.config2_textured(width=SIZE, height=SIZE, segments=10, rings=7, extended=True,
                                texture=source).draws[0]
    d.texture = (SIZE, SIZE, source, False)
    d.uniform = scenes.perspective_view(50.0 + k, 1.0, 0.1, 10.0, 2.0)
    d.cull_mode = wgc.CULL_NONE
    return d


class Targets:
    """Three colour targets with a depth texture each, and passes on them:
    ("draw", target) blends onto what is there, ("sample", source, target)
    draws a mesh textured with another target's contents."""

    def __init__(self, steps):
        self.dev = wgc.Device(0, wgc.SEMANTICS_EXTENDED)
        self.keep, cache = [], {}
        self.res = [SimpleNamespace(color=self.dev.create_texture(SIZE, SIZE, wgc.RGBA8_UNORM),
                                    depth=self.dev.create_texture(SIZE, SIZE, wgc.DEPTH32_FLOAT)) for _ in range(3)]
        for i, r in enumerate(self.res):
            cache[("tex", SIZE, SIZE, b"target %d" % i, False)] = r.color
        self.buffers = []
        for k, s in enumerate(steps):
            if s[0] == "draw":
                spec = scenes.PassSpec(SIZE, SIZE, draws=[blended(200 + 700 * (k % 3), 8100 + k)],
                                       clear_color=None if k > 2 else (0.2, 0.1 * k, 0.0, 1.0),
                                       semantics=wgc.SEMANTICS_EXTENDED)
                res = SimpleNamespace(color=self.res[s[1]].color, depth=None)
            else:
                spec = scenes.PassSpec(SIZE, SIZE, draws=[textured(b"target %d" % s[1], k)], clear_color=None,
                                       has_depth=True, clear_depth=1.0, semantics=wgc.SEMANTICS_EXTENDED)
                res = self.res[s[2]]
            enc = self.dev.create_command_encoder()
            runner.record_pass(self.dev, enc, spec, res, self.keep, cache)
            self.buffers.append(enc.finish())

    def read(self):
        self.dev.poll()
        return [np.frombuffer(r.color.read(), np.uint8) for r in self.res]


STEPS = [("draw", 0), ("draw", 1), ("draw", 2), ("sample", 0, 1), ("sample", 1, 2), ("draw", 0), ("sample", 2, 0),
         ("draw", 1), ("draw", 1), ("sample", 1, 0), ("sample", 1, 2), ("draw", 1), ("sample", 0, 1), ("draw", 2)]


@pytest.mark.parametrize("repeat", [1, 6])
@pytest.mark.parametrize("extra", ["none", "write", "timestamp", "copy", "group", "read"])
def test_dependent_submissions(repeat, extra):
    announce(f"dependent submissions {extra} x{repeat}")
    noise = np.random.default_rng(5).integers(0, 256, SIZE * SIZE * 4, dtype=np.uint8).tobytes()

    def run(wait):
        t = Targets(STEPS)
        enc = t.dev.create_command_encoder()
        buf = t.dev.create_buffer(SIZE * 512)
        enc.copy_texture_to_buffer(t.res[2].color, (0, 0), buf, 0, 512, SIZE, SIZE)
        enc.copy_buffer_to_texture(buf, 0, 512, t.res[0].color, (0, 0), SIZE, SIZE)
        copy = enc.finish()
        seen = []
        for n in range(repeat):
            for k, cb in enumerate(t.buffers):
                t.dev.submit([cb])
                if k % 4 == 2:
                    if extra == "write":
                        t.dev.write_texture(t.res[(k // 4) % 3].color, noise)
                    elif extra == "timestamp":
                        t.dev.timestamp(k)
                    elif extra == "copy":
                        t.dev.submit([copy])
                    elif extra == "group":
                        t.dev.submit([t.buffers[5], t.buffers[9], t.buffers[4]])
                    elif extra == "read":
                        seen.append(np.frombuffer(t.res[k % 3].color.read(), np.uint8))
                if wait:
                    t.dev.poll()
        return seen + t.read()

    for got, want in zip(run(False), run(True)):
        np.testing.assert_array_equal(got, want)


def test_independent_submissions_from_threads():
    """Four threads, each its own targets; every pass against the oracle."""
    announce("independent submissions from threads")
    dev = wgc.Device(0, wgc.SEMANTICS_EXTENDED)
    specs = [scenes.PassSpec(60 + 41 * i, 120 - 13 * i, clear_color=(0.1, 0.2, 0.3, 1.0),
                             draws=[blended(n, 8200 + i, 60 + 41 * i, 120 - 13 * i)],
                             semantics=wgc.SEMANTICS_EXTENDED) for i, n in enumerate((3, 500, 2000, 9000))]
    passes = [runner.PreparedPass(dev, s) for s in specs]
    threads = [threading.Thread(target=lambda p=p: [p.submit() for _ in range(25)]) for p in passes]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    fragments = 25 * sum(bridge.render(s).fragments for s in specs)
    dev.poll()
    assert dev.totals()[0] == fragments
    for p, s in zip(passes, specs):
        ref = bridge.render(s)
        np.testing.assert_array_equal(p.results()[0].color, ref.color)


def test_written_between_submissions():
    """A vertex buffer written between submissions on several targets."""
    announce("written between submissions")
    dev = wgc.Device(0, wgc.SEMANTICS_EXTENDED)
    datas = [random_clip_triangles(300, 8300 + i, SIZE, SIZE, alpha=(0.2, 0.8)) for i in range(6)]
    specs = [scenes.PassSpec(SIZE, SIZE, clear_color=(0.0, 0.0, 0.0, 1.0),
                             draws=[clip_color_draw(v, depth=None, blend=wgc.BLEND_ALPHA)],
                             semantics=wgc.SEMANTICS_EXTENDED) for v in datas]
    cache, keep = {}, []
    vb = dev.create_buffer_init(specs[0].draws[0].vertex_data)
    cache[("buf", specs[0].draws[0].vertex_data)] = vb
    res = [runner._PassResources(dev, specs[0], keep) for _ in specs]
    buffers = []
    for r in res:
        enc = dev.create_command_encoder()
        runner.record_pass(dev, enc, specs[0], r, keep, cache)
        buffers.append(enc.finish())
    for _ in range(3):
        for s, cb in zip(specs, buffers):
            dev.write_buffer(vb, 0, s.draws[0].vertex_data)
            dev.submit([cb])
            dev.submit([cb])
    dev.poll()
    for s, r in zip(specs, res):
        np.testing.assert_array_equal(r.read()[0], bridge.render(s).color)


def test_heap_targets_reused_between_lanes():
    """Targets from a heap that is full with four of them: each is released
    as soon as its picture has been copied, and the next takes its place while
    passes on other targets run."""
    announce("heap targets reused between lanes")
    dev = wgc.Device(0, wgc.SEMANTICS_EXTENDED)
    heap = dev.create_heap(4 * SIZE * SIZE * 4)
    specs = [scenes.PassSpec(SIZE, SIZE, clear_color=(0.1 * i, 0.2, 0.3, 1.0), draws=[blended(150 + 400 * i, 8400 + i)],
                             semantics=wgc.SEMANTICS_EXTENDED) for i in range(5)]
    refs = [bridge.render(s).color for s in specs]
    keep, cache, out = [], {}, []
    for n in range(40):
        target = heap.create_texture(SIZE, SIZE, wgc.RGBA8_UNORM)
        if target is None:      # full until the last submissions of released ones have executed
            dev.poll()
            target = heap.create_texture(SIZE, SIZE, wgc.RGBA8_UNORM)
        enc = dev.create_command_encoder()
        runner.record_pass(dev, enc, specs[n % 5], SimpleNamespace(color=target, depth=None), keep, cache)
        draw = enc.finish()
        dev.submit([draw])
        if n % 3 == 0:
            dev.submit([draw])
        enc = dev.create_command_encoder()
        buf = dev.create_buffer(SIZE * 512)
        enc.copy_texture_to_buffer(target, (0, 0), buf, 0, 512, SIZE, SIZE)
        dev.submit([enc.finish()])
        out.append(buf)
        target.release()
    dev.poll()
    for n, buf in enumerate(out):
        got = np.frombuffer(buf.read(), np.uint8).reshape(SIZE, 512)[:, :SIZE * 4].reshape(SIZE, SIZE, 4)
        np.testing.assert_array_equal(got, refs[n % 5])


def test_mapped_between_submissions():
    """A vertex buffer written through a mapping between submissions on
    several targets, some of them running on the other lane."""
    announce("mapped between submissions")
    dev = wgc.Device(0, wgc.SEMANTICS_EXTENDED)
    datas = [random_clip_triangles(300, 8500 + i, SIZE, SIZE, alpha=(0.2, 0.8)) for i in range(6)]
    specs = [scenes.PassSpec(SIZE, SIZE, clear_color=(0.0, 0.0, 0.0, 1.0),
                             draws=[clip_color_draw(v, depth=None, blend=wgc.BLEND_ALPHA)],
                             semantics=wgc.SEMANTICS_EXTENDED) for v in datas]
    cache, keep = {}, []
    data = specs[0].draws[0].vertex_data
    vb = dev.create_buffer_init(data)
    cache[("buf", data)] = vb
    others = [runner.PreparedPass(dev, scenes.PassSpec(SIZE, SIZE, draws=[blended(900, 8600 + i)],
                                                       semantics=wgc.SEMANTICS_EXTENDED)) for i in range(2)]
    res = [runner._PassResources(dev, specs[0], keep) for _ in specs]
    buffers = []
    for r in res:
        enc = dev.create_command_encoder()
        runner.record_pass(dev, enc, specs[0], r, keep, cache)
        buffers.append(enc.finish())
    for _ in range(3):
        for s, cb in zip(specs, buffers):
            vb.map_async(wgc.MAP_WRITE)
            dev.poll()
            np.frombuffer(vb.get_mapped_range(), np.uint8)[:] = np.frombuffer(s.draws[0].vertex_data, np.uint8)
            for o in others:
                o.submit()
            vb.unmap()
            for o in others:
                o.submit()
            dev.submit([cb])
            dev.submit([cb])
    dev.poll()
    for s, r in zip(specs, res):
        np.testing.assert_array_equal(r.read()[0], bridge.render(s).color)
