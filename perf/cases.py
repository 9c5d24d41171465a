"""The render work whose speed is measured: frames, overdraw, scenes, lines,
batches and requests, each through the package's public interface (`wgc`).

A case is a dict of plain values.  Its `kind` names what a program does:

  mesh      one command buffer with one draw of an indexed mesh, submitted
            again every frame (targets and mesh stay on the GPU)
  frame     the same draw the way a wgpu program drives it: the camera
            uniform written, the pass recorded anew, one submission a frame
  image     an off-screen picture: a recorded pass, the texture copied to a
            buffer, the buffer mapped and its bytes in host memory
  triangles clip-space triangles of a particle / overdraw layer, overwriting
            or blended (src-over) in API order
  scene     one pass with many draws: objects with their own meshes and
            camera matrices, sharing the target and its depth
  lines     a line list (wireframes, plots), depth-tested or blended
  batch     many small independent passes in one command buffer
  serve     requests that arrive with their own sizes: targets and uniforms
            from a heap, passes recorded and submitted together

A pass leaves its results in textures on the GPU, which a program presents
or samples and does not copy to the host.  `run` therefore returns them as a
mapping that reads a texture back when it is looked at; only `image`, whose
product is host memory, copies inside the pass.
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import numpy as np

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "wgpu-cpu_amd"))

import wgc  # noqa: E402
from wgc import runner, scenes  # noqa: E402

CLEAR = (0.1, 0.2, 0.3, 1.0)
TEXTURE = 1024          # side of the sampled texture
MESHES = 8              # resident meshes of a batch or a server
SCENE_MESHES = 4        # different meshes among a scene's objects


def listed():
    return [
        # a plain window of one small object, drawn anew each frame: launches and host work count
        {"name": "frame 256x256", "kind": "frame", "w": 256, "h": 256, "tris": 960, "textured": False, "wgsl": False},
        # a thumbnail or golden image: rendered, copied, mapped, read; an odd size
        {"name": "image 611x403", "kind": "image", "w": 611, "h": 403, "tris": 5000, "textured": True, "wgsl": True},
        # the headline frame: bilinear, perspective-correct, sRGB-decoded texturing at 1080p
        {"name": "mesh 1080p extended", "kind": "mesh", "w": 1920, "h": 1080, "tris": 65024, "textured": True,
         "ext": True, "wgsl": False},
        # the same frame as the reference shades it, with the program's own WGSL shaders
        {"name": "mesh 1080p wgsl", "kind": "mesh", "w": 1920, "h": 1080, "tris": 65024, "textured": True,
         "ext": False, "wgsl": True},
        # the largest frame: 4K, half a million triangles
        {"name": "mesh 4K", "kind": "mesh", "w": 3840, "h": 2160, "tris": 500000, "textured": True, "ext": True,
         "wgsl": False},
        # overdraw in API order, overwriting (the reference's colour write)
        {"name": "triangles overwrite 200k", "kind": "triangles", "w": 2560, "h": 2440, "n": 200000, "blend": False},
        # the same layer blended
        {"name": "triangles blend 200k", "kind": "triangles", "w": 2560, "h": 2440, "n": 200000, "blend": True},
        # a scene of objects in one pass, at a common laptop size
        {"name": "scene 24 objects 1366x768", "kind": "scene", "w": 1366, "h": 768, "objects": 24, "tris": 3000,
         "textured": True, "wgsl": True},
        # a wireframe or plot: thousands of depth-tested lines
        {"name": "lines depth 20k", "kind": "lines", "w": 1920, "h": 1080, "n": 20000, "length": 80, "blend": False},
        # translucent lines (graph edges, trails)
        {"name": "lines blend 4k", "kind": "lines", "w": 1600, "h": 901, "n": 4000, "length": 100, "blend": True},
        # many independent passes in one submission
        {"name": "batch 256", "kind": "batch", "passes": 256, "max_side": 1024, "max_tris": 50000},
        # a few requests of a server, as they arrive
        {"name": "serve 6 requests", "kind": "serve", "requests": 6, "max_side": 1024, "max_tris": 50000},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["mesh", "mesh", "frame", "image", "triangles", "triangles", "scene", "lines", "batch", "serve"])
    if kind in ("mesh", "frame", "image"):
        big = kind == "mesh"
        c = {"kind": kind, "w": _log(rng, 64, 3840 if big else 1920), "h": _log(rng, 64, 2160 if big else 1080),
             "tris": _log(rng, 100, 500000 if big else 50000), "textured": rng.random() < 0.6,
             "wgsl": rng.random() < 0.5}
        if big:
            c["ext"] = rng.random() < 0.5
        return c
    if kind == "triangles":
        return {"kind": kind, "w": _log(rng, 256, 2560), "h": _log(rng, 256, 2440), "n": _log(rng, 500, 200000),
                "blend": rng.random() < 0.5}
    if kind == "scene":
        return {"kind": kind, "w": _log(rng, 256, 1920), "h": _log(rng, 256, 1080), "objects": rng.randint(2, 24),
                "tris": _log(rng, 100, 20000), "textured": rng.random() < 0.5, "wgsl": rng.random() < 0.5}
    if kind == "lines":
        blend = rng.random() < 0.5
        length = _log(rng, 8, 200)
        most = 400000 // length if blend else 1600000 // length
        return {"kind": kind, "w": _log(rng, 256, 1920), "h": _log(rng, 256, 1080),
                "n": _log(rng, 200, min(20000, most)), "length": length, "blend": blend}
    if kind == "batch":
        return {"kind": kind, "passes": _log(rng, 4, 256), "max_side": _log(rng, 128, 1024),
                "max_tris": _log(rng, 1000, 50000)}
    return {"kind": kind, "requests": rng.randint(1, 12), "max_side": _log(rng, 128, 1024),
            "max_tris": _log(rng, 1000, 50000)}


# ------------------------------------------------------------------
# inputs, from the seed alone
# ------------------------------------------------------------------

def _rng(seed, *more):
    return np.random.default_rng([int(seed) & 0xFFFFFFFF, *more])


def _shape(tris):
    """(segments, rings) of a sphere of about `tris` triangles; the 256x128 one has 65,024."""
    rings = max(3, int(round(math.sqrt(tris / 4.0))) + (1 if tris > 2000 else 0))
    return 2 * rings, rings


def _sphere(segments, rings, rng):
    """A UV sphere of radius about 1, radially displaced by a few smooth
    waves; outward faces wind counter-clockwise.  Positions, uv, u32 indices."""
    theta = np.pi * np.arange(rings + 1) / rings
    phi = 2.0 * np.pi * np.arange(segments + 1) / segments
    st, ct = np.sin(theta)[:, None], np.cos(theta)[:, None]
    pos = np.stack([st * np.cos(phi), np.broadcast_to(ct, (rings + 1, segments + 1)), -st * np.sin(phi)], -1)
    pos = pos.reshape(-1, 3)
    bump = np.zeros(len(pos))
    for _ in range(5):
        bump += np.sin(pos @ rng.normal(0.0, 4.0, 3) + rng.uniform(0.0, 6.28))
    pos = pos * (1.0 + 0.01 * bump)[:, None]
    uv = np.stack(np.meshgrid(np.arange(segments + 1) / segments, np.arange(rings + 1) / rings), -1).reshape(-1, 2)
    r, s = np.meshgrid(np.arange(rings), np.arange(segments), indexing="ij")
    a = r * (segments + 1) + s
    c = a + segments + 1
    two = np.stack([np.stack([a, c, a + 1], -1), np.stack([a + 1, c, c + 1], -1)], 2)
    keep = np.stack([r != 0, r != rings - 1], -1)     # one triangle per segment at the poles
    return pos, uv, two[keep].astype(np.uint32).reshape(-1)


def _camera(w, h, yaw, at=(0.0, 0.0), scale=1.0):
    """Projection * view * model as column-major f32: an object of `scale`
    turned by `yaw` at (x, y) units from the middle of the view."""
    f, near, far = 1.0 / math.tan(math.radians(30.0)), 0.1, 10.0
    proj = np.array([[f * h / w, 0, 0, 0], [0, f, 0, 0], [0, 0, far / (near - far), near * far / (near - far)],
                     [0, 0, -1, 0]])
    c, s = math.cos(yaw) * scale, math.sin(yaw) * scale
    model = np.array([[c, 0, s, at[0]], [0, scale, 0, at[1]], [-s, 0, c, -3.0], [0, 0, 0, 1]])
    return (proj @ model).astype(np.float32)


def _texture(seed):
    rng = _rng(seed, 77)
    y, x = np.mgrid[0:TEXTURE, 0:TEXTURE]
    t = np.full((TEXTURE, TEXTURE, 4), 255, np.int16)
    t[..., :3] = (((x // 32 + y // 32) % 2) * 223)[..., None] + rng.integers(0, 33, (TEXTURE, TEXTURE, 3), np.int16)
    return t.astype(np.uint8).tobytes()


def _mesh(seed, number, tris, textured):
    """(vertex array, attributes, indices) of a mesh: position vec4 and uv or a vec3 colour."""
    rng = _rng(seed, 1, number)
    pos, uv, idx = _sphere(*_shape(tris), rng)
    more = uv if textured else rng.random((len(pos), 3))
    vb = np.concatenate([pos, np.ones((len(pos), 1)), more], 1).astype(np.float32)
    return vb, idx


def _mesh_draw(vb, idx, matrix, textured, texture, ext, wgsl):
    program = wgc.PROGRAM_MVP_TEXTURE if textured else wgc.PROGRAM_MVP_COLOR
    interp = wgc.INTERP_PERSPECTIVE if ext else wgc.INTERP_LINEAR
    return scenes.DrawSpec(
        program=program, interp=interp, vertex_data=vb.tobytes(), vertex_stride=vb.shape[1] * 4,
        attributes=[(wgc.FLOAT32X4, 0, 0), (wgc.FLOAT32X2 if textured else wgc.FLOAT32X3, 16, 1)],
        index_data=idx.tobytes(), uniform=matrix.T.tobytes(),
        texture=(TEXTURE, TEXTURE, texture, True) if textured else None,
        filter=wgc.FILTER_LINEAR if ext else wgc.FILTER_NEAREST, cull_mode=wgc.CULL_BACK, depth=(wgc.LESS, True),
        count=len(idx), wgsl=scenes.wgsl_source(program, interp, 0 if textured else 3) if wgsl else None)


def _triangles(case, seed):
    """Equilateral triangles, log-normal areas of median 40 px, any turn, RGBA of alpha 0.1-0.9."""
    rng, n, w, h = _rng(seed, 2), case["n"], case["w"], case["h"]
    area = np.clip(40.0 * np.exp(rng.standard_normal(n)), 4.0, 400.0)
    radius = np.sqrt(4.0 * area / math.sqrt(3.0)) / math.sqrt(3.0)
    ang = rng.uniform(0.0, 2.0 * np.pi, n)[:, None] + np.array([0.0, 2.0, 4.0]) * np.pi / 3.0
    vb = np.zeros((n, 3, 8), np.float32)
    vb[:, :, 0] = (rng.uniform(0, w, n)[:, None] + radius[:, None] * np.cos(ang)) / w * 2.0 - 1.0
    vb[:, :, 1] = 1.0 - (rng.uniform(0, h, n)[:, None] + radius[:, None] * np.sin(ang)) / h * 2.0
    vb[:, :, 2], vb[:, :, 3] = 0.5, 1.0
    vb[:, :, 4:7] = rng.random((n, 1, 3))
    vb[:, :, 7] = 0.1 + 0.8 * rng.random((n, 1))
    return vb.reshape(-1, 8)


def _lines(case, seed):
    """Lines of about `length` pixels anywhere on the target, RGBA of alpha 0.1-0.9, depths across the range."""
    rng, n, w, h = _rng(seed, 3), case["n"], case["w"], case["h"]
    mid = rng.uniform(0.0, 1.0, (n, 2)) * (w, h)
    ang = rng.uniform(0.0, 2.0 * np.pi, n)
    half = 0.5 * case["length"] * rng.uniform(0.5, 1.5, n)
    step = np.stack([half * np.cos(ang), half * np.sin(ang)], -1)
    xy = np.stack([mid - step, mid + step], 1)
    vb = np.zeros((n, 2, 8), np.float32)
    vb[:, :, 0] = xy[..., 0] / w * 2.0 - 1.0
    vb[:, :, 1] = 1.0 - xy[..., 1] / h * 2.0
    vb[:, :, 2] = rng.uniform(0.05, 0.95, (n, 2))
    vb[:, :, 3] = 1.0
    vb[:, :, 4:7] = rng.random((n, 1, 3))
    vb[:, :, 7] = 0.1 + 0.8 * rng.random((n, 1))
    return vb.reshape(-1, 8)


def _objects(case, seed):
    """A scene's objects: (mesh number, matrix) in draw order."""
    rng = _rng(seed, 4)
    aspect = case["w"] / case["h"]
    out = []
    for _ in range(case["objects"]):
        at = (rng.uniform(-1.2, 1.2) * aspect, rng.uniform(-1.2, 1.2))
        m = _camera(case["w"], case["h"], rng.uniform(0, 6.28), at, rng.uniform(0.2, 0.6))
        out.append((int(rng.integers(SCENE_MESHES)), m))
    return out


def _passes(case, seed):
    """Passes of a batch or requests of a server: (w, h, mesh number, matrix).
    Odd mesh numbers are textured.  Sizes and meshes belong to the case, the
    cameras to the seed."""
    n = case.get("passes") or case["requests"]
    size, rng = _rng(n, 5, case["max_side"]), _rng(seed, 6)
    out = []
    for _ in range(n):
        w, h = (int(round(math.exp(size.uniform(math.log(64), math.log(case["max_side"]))))) for _ in range(2))
        out.append((w, h, int(size.integers(MESHES)), _camera(w, h, rng.uniform(0, 6.28))))
    return out


def _pool(case, seed):
    """The resident meshes of a batch or a server, 100 triangles to the case's most."""
    sizes = np.exp(np.linspace(math.log(100), math.log(case["max_tris"]), MESHES))
    return [_mesh(seed, k, float(sizes[k]), k % 2 == 1) for k in range(MESHES)]


# ------------------------------------------------------------------
# programs
# ------------------------------------------------------------------

class Images(dict):
    """Named textures of a pass; each is read back when it is looked at."""

    def __getitem__(self, name):
        return dict.__getitem__(self, name)()


def _read(texture):
    data = texture.read()
    if texture.format == wgc.DEPTH32_FLOAT:
        return np.frombuffer(data, np.float32).reshape(texture.height, texture.width)
    return np.frombuffer(data, np.uint8).reshape(texture.height, texture.width, 4)


def _images(pairs):
    """Images of the passes' (colour, depth) textures: one array for one pass, else all passes' texels in a row."""
    def whole(k):
        def read():
            if len(pairs) == 1:
                return _read(pairs[0][k])
            return np.concatenate([_read(p[k]).reshape(-1) for p in pairs])
        return read
    return Images({name: whole(k) for k, name in ((0, "color"), (1, "depth")) if pairs[0][k] is not None})


_DEVICES = {}


def _device(ext):
    """A program keeps one device for its life."""
    sem = wgc.SEMANTICS_EXTENDED if ext else wgc.SEMANTICS_REFERENCE
    if sem not in _DEVICES:
        _DEVICES[sem] = wgc.Device(0, sem)
    return _DEVICES[sem]


def _is_ext(case):
    return bool(case.get("ext") or case.get("blend"))


def _prepared(dev, specs):
    pp = runner.PreparedPasses(dev, specs)
    return {"submit": pp.submit, "keep": pp, "images": _images([(r.color, r.depth) for r in pp.res])}


def _resident(dev, mesh, textured, wgsl, texture, depth_format=wgc.DEPTH32_FLOAT):
    """Pipeline and buffers of a mesh that a program draws again and again."""
    vb, idx = mesh
    program = wgc.PROGRAM_MVP_TEXTURE if textured else wgc.PROGRAM_MVP_COLOR
    module = (dev.create_shader_module_wgsl(scenes.wgsl_source(program, wgc.INTERP_LINEAR, 0 if textured else 3))
              if wgsl else dev.create_shader_module_builtin(program, wgc.INTERP_LINEAR))
    attrs = [(wgc.FLOAT32X4, 0, 0), (wgc.FLOAT32X2 if textured else wgc.FLOAT32X3, 16, 1)]
    out = {"pipeline": dev.create_render_pipeline(module, [(vb.shape[1] * 4, wgc.STEP_VERTEX, attrs)],
                                                  cull_mode=wgc.CULL_BACK, depth=(wgc.LESS, True)),
           "module": module, "vertices": dev.create_buffer_init(vb.tobytes()),
           "indices": dev.create_buffer_init(idx.tobytes()), "count": len(idx), "bind1": None}
    if textured:
        out["bind1"] = dev.create_bind_group([(0, texture[0]), (1, texture[1])])
    return out


def _sampled(dev, seed):
    tex = dev.create_texture(TEXTURE, TEXTURE, wgc.RGBA8_UNORM_SRGB)
    dev.write_texture(tex, _texture(seed))
    return tex, dev.create_sampler(wgc.REPEAT, wgc.REPEAT)


def _record(enc, mesh, color, depth, bind0):
    rp = enc.begin_render_pass(color=color, clear_color=CLEAR, depth=depth, clear_depth=1.0)
    rp.set_pipeline(mesh["pipeline"])
    rp.set_bind_group(0, bind0)
    if mesh["bind1"] is not None:
        rp.set_bind_group(1, mesh["bind1"])
    rp.set_vertex_buffer(0, mesh["vertices"])
    rp.set_index_buffer(mesh["indices"], wgc.INDEX_UINT32)
    rp.draw_indexed(range(0, mesh["count"]))
    rp.end()


def prepare(case, seed):
    kind, dev = case["kind"], _device(_is_ext(case))
    s = {"case": case, "dev": dev}
    if kind == "mesh":
        w, h, textured = case["w"], case["h"], case["textured"]
        vb, idx = _mesh(seed, 0, case["tris"], textured)
        d = _mesh_draw(vb, idx, _camera(w, h, _rng(seed).uniform(0, 6.28)), textured,
                       _texture(seed) if textured else None, case["ext"], case["wgsl"])
        s.update(_prepared(dev, [scenes.PassSpec(w, h, clear_color=CLEAR, has_depth=True, draws=[d],
                                                 semantics=dev.semantics)]))
    elif kind in ("frame", "image"):
        w, h, textured = case["w"], case["h"], case["textured"]
        s["mesh"] = _resident(dev, _mesh(seed, 0, case["tris"], textured), textured, case["wgsl"],
                              _sampled(dev, seed) if textured else None)
        s["matrix"] = _camera(w, h, _rng(seed).uniform(0, 6.28)).T.tobytes()
        s["uniform"] = dev.create_buffer(64)
        s["bind0"] = dev.create_bind_group([(0, s["uniform"])])
        s["color"] = dev.create_texture(w, h, wgc.RGBA8_UNORM)
        s["depth"] = dev.create_texture(w, h, wgc.DEPTH32_FLOAT)
        s["images"] = _images([(s["color"], s["depth"])])
        if kind == "image":
            s["pitch"] = (w * 4 + 255) // 256 * 256
            s["buffer"] = dev.create_buffer(s["pitch"] * h)
    elif kind in ("triangles", "lines"):
        vb = _triangles(case, seed) if kind == "triangles" else _lines(case, seed)
        depth = kind == "lines" and not case["blend"]
        d = scenes.DrawSpec(program=wgc.PROGRAM_CLIP_COLOR, vertex_data=vb.tobytes(), vertex_stride=32,
                            attributes=[(wgc.FLOAT32X4, 0, 0), (wgc.FLOAT32X4, 16, 1)], count=len(vb),
                            topology=wgc.LINE_LIST if kind == "lines" else wgc.TRIANGLE_LIST,
                            blend=wgc.BLEND_ALPHA if case["blend"] else wgc.BLEND_REPLACE,
                            depth=(wgc.LESS, True) if depth else None)
        s.update(_prepared(dev, [scenes.PassSpec(case["w"], case["h"], clear_color=CLEAR, has_depth=depth, draws=[d],
                                                 semantics=dev.semantics)]))
    elif kind == "scene":
        texture = _texture(seed) if case["textured"] else None
        meshes = [_mesh(seed, k, case["tris"] / 2.0 ** k, case["textured"]) for k in range(SCENE_MESHES)]
        draws = [_mesh_draw(*meshes[k], m, case["textured"], texture, False, case["wgsl"])
                 for k, m in _objects(case, seed)]
        s.update(_prepared(dev, [scenes.PassSpec(case["w"], case["h"], clear_color=CLEAR, has_depth=True,
                                                 draws=draws)]))
    elif kind == "batch":
        pool, texture = _pool(case, seed), _texture(seed)
        specs = [scenes.PassSpec(w, h, clear_color=CLEAR, has_depth=True,
                                 draws=[_mesh_draw(*pool[k], m, k % 2 == 1, texture, False, False)])
                 for w, h, k, m in _passes(case, seed)]
        s.update(_prepared(dev, specs))
    else:
        texture = _sampled(dev, seed)
        s["pool"] = [_resident(dev, m, k % 2 == 1, False, texture) for k, m in enumerate(_pool(case, seed))]
        s["heap"] = dev.create_heap(1 << 30)
        s["requests"] = [(w, h, k, m.T.tobytes()) for w, h, k, m in _passes(case, seed)]
    return s


def _serve(s):
    """Admits the requests (targets and uniforms from the heap), records and
    submits them together.  The last call's targets were handed over before
    and go back to the heap with their handles."""
    dev, heap = s["dev"], s["heap"]
    enc = dev.create_command_encoder()
    targets, keep = [], []
    for w, h, k, matrix in s["requests"]:
        color, depth = heap.create_texture(w, h, wgc.RGBA8_UNORM), heap.create_texture(w, h, wgc.DEPTH32_FLOAT)
        uniform = heap.create_buffer(64)
        dev.write_buffer(uniform, 0, matrix)
        bind0 = dev.create_bind_group([(0, uniform)])
        _record(enc, s["pool"][k], color, depth, bind0)
        targets.append((color, depth))
        keep += [uniform, bind0]
    dev.submit([enc.finish()])
    return _images(targets)


def run(state):
    s, kind = state, state["case"]["kind"]
    if kind == "serve":
        return _serve(s)
    if kind not in ("frame", "image"):
        s["submit"]()
        return s["images"]
    dev, case = s["dev"], s["case"]
    dev.write_buffer(s["uniform"], 0, s["matrix"])
    enc = dev.create_command_encoder()
    _record(enc, s["mesh"], s["color"], s["depth"], s["bind0"])
    if kind == "frame":
        dev.submit([enc.finish()])
        return s["images"]
    w, h, buf = case["w"], case["h"], s["buffer"]
    enc.copy_texture_to_buffer(s["color"], (0, 0), buf, 0, s["pitch"], w, h)
    dev.submit([enc.finish()])
    buf.map_async(wgc.MAP_READ)
    dev.poll()
    rows = np.frombuffer(buf.get_mapped_range(), np.uint8).reshape(h, s["pitch"])
    picture = rows[:, :w * 4].reshape(h, w, 4).copy()
    buf.unmap()
    return {"color": picture}


# ------------------------------------------------------------------
# what a pass cannot do without
# ------------------------------------------------------------------

def _mesh_work(w, h, tris, textured):
    """Bytes and operations of a mesh pass: targets written, mesh and texture
    read once; 32 operations a vertex, about 100 a triangle, 60 a pixel of the disc."""
    segments, rings = _shape(tris)
    verts, prims = (segments + 1) * (rings + 1), 2 * segments * (rings - 1)
    pixels = min(w * h, 0.26 * math.pi * h * h)
    return (8.0 * w * h + verts * (24 if textured else 28) + prims * 12 + 64,
            32.0 * verts + 100.0 * prims + 60.0 * pixels)


def work(case):
    kind = case["kind"]
    tex = 4.0 * TEXTURE * TEXTURE
    if kind in ("mesh", "frame", "image"):
        b, f = _mesh_work(case["w"], case["h"], case["tris"], case["textured"])
        if kind == "image":
            b += 8.0 * case["w"] * case["h"]
        return {"bytes": b + (tex if case["textured"] else 0), "flops": f}
    if kind == "triangles":
        return {"bytes": 4.0 * case["w"] * case["h"] + 96.0 * case["n"], "flops": case["n"] * (100.0 + 60.0 * 60.0)}
    if kind == "lines":
        return {"bytes": (4.0 if case["blend"] else 8.0) * case["w"] * case["h"] + 64.0 * case["n"],
                "flops": case["n"] * (60.0 + 30.0 * case["length"])}
    if kind == "scene":
        b = 8.0 * case["w"] * case["h"] + (tex if case["textured"] else 0) + 64.0 * case["objects"]
        f = 60.0 * case["w"] * case["h"] * 0.5
        for k in range(SCENE_MESHES):
            mb, mf = _mesh_work(0, 0, case["tris"] / 2.0 ** k, case["textured"])
            b, f = b + mb, f + mf * case["objects"] / SCENE_MESHES
        return {"bytes": b, "flops": f}
    sizes = np.exp(np.linspace(math.log(100), math.log(case["max_tris"]), MESHES))
    b, f = tex, 0.0
    for w, h, k, _ in _passes(case, 0):
        pb, pf = _mesh_work(w, h, float(sizes[k]), k % 2 == 1)
        b, f = b + pb, f + pf
    return {"bytes": b, "flops": f}


def tolerance(case):
    """The executor's arithmetic is fixed operation by operation (binary32,
    one rounding each, a defined order): another correct implementation gives
    the same bits."""
    return "exact"


# ------------------------------------------------------------------
# the depths in 64 bits
# ------------------------------------------------------------------

def _clip(vb, idx, matrix):
    p = vb[idx, :4].astype(np.float64) if idx is not None else vb[:, :4].astype(np.float64)
    return p @ matrix.astype(np.float64).T if matrix is not None else p


def _expand(counts):
    """(owner, place) of every item when owner k has counts[k] of them."""
    owner = np.repeat(np.arange(len(counts)), counts)
    return owner, np.arange(len(owner)) - np.repeat(np.cumsum(counts) - counts, counts)


def _depth_triangles(depth, clip):
    """Less-tested depths of back-face-culled triangles (N, 3, 4) into `depth`
    (h, w): integer scanlines between truncated vertices, depth at the pixel
    corner.  Triangles across a side of the view are cut by pixel, not by
    the clipper."""
    h, w = depth.shape
    ndc = clip[..., :3] / clip[..., 3:]
    a, b, c = ndc[:, 0], ndc[:, 1], ndc[:, 2]
    ndc = ndc[(b - a)[:, 0] * (c - a)[:, 1] - (b - a)[:, 1] * (c - a)[:, 0] > 0]
    x, y, z = (ndc[..., 0] + 1) * 0.5 * w, (1 - ndc[..., 1]) * 0.5 * h, ndc[..., 2]
    ix, iy = np.floor(x).astype(np.int64), np.floor(y).astype(np.int64)
    order = np.argsort(iy, 1, kind="stable")
    sx, sy = np.take_along_axis(ix, order, 1), np.take_along_axis(iy, order, 1)
    last = np.where((sy[:, 2] == sy[:, 1]) & (sy[:, 1] != sy[:, 0]), sy[:, 1] - 1, sy[:, 2])
    first = np.maximum(sy[:, 0], 0)
    tri, row = _expand(np.maximum(np.minimum(last, h - 1) - first + 1, 0))
    py = row + first[tri]
    (ax, bx, cx), (ay, by, cy) = sx[tri].T, sy[tri].T

    def edge(x0, y0, x1, y1):
        q = (x1 - x0) * (py - y0)
        d = np.where(y1 == y0, 1, y1 - y0)
        return x0 + np.sign(q) * (np.abs(q) // d)

    one, two = edge(ax, ay, cx, cy), np.where(py < by, edge(ax, ay, bx, by), edge(bx, by, cx, cy))
    flat = cy == ay
    lo = np.where(flat, np.minimum(np.minimum(ax, bx), cx), np.minimum(one, two))
    hi = np.where(flat, np.maximum(np.maximum(ax, bx), cx), np.maximum(one, two))
    lo, hi = np.maximum(lo, 0), np.minimum(hi, w - 1)
    span, place = _expand(np.maximum(hi - lo + 1, 0))
    px, py, tri = lo[span] + place, py[span], tri[span]
    (x0, x1, x2), (y0, y1, y2), (z0, z1, z2) = x[tri].T, y[tri].T, z[tri].T
    total = (x1 - x0) * (y2 - y0) - (y1 - y0) * (x2 - x0)
    l1 = ((px - x0) * (y2 - y0) - (py - y0) * (x2 - x0)) / total
    l2 = ((x1 - x0) * (py - y0) - (y1 - y0) * (px - x0)) / total
    np.minimum.at(depth, (py, px), z0 + l1 * (z1 - z0) + l2 * (z2 - z0))


def _depth_lines(depth, clip):
    """Less-tested depths of lines (N, 2, 4): cut to the view, then one
    fragment a step of the major axis, its last left out.  The cut's end
    points and coefficients go into each other as the executor's do."""
    h, w = depth.shape
    p, q = clip[:, 0], clip[:, 1]
    side = np.array([[1, 0, 0, 1], [-1, 0, 0, 1], [0, 1, 0, 1], [0, -1, 0, 1], [0, 0, 1, 0], [0, 0, -1, 1.0]])
    dp, dq = p @ side.T, q @ side.T
    cut = dp / np.where(dp == dq, 1.0, dp - dq)
    a0 = np.where(dp < 0, cut, 0.0).max(1)[:, None]
    a1 = np.where((dq < 0) & (dp >= 0), cut, 1.0).min(1)[:, None]
    p = p * (1 - a0) + q * a0
    q = p * (1 - a1) + q * a1
    ok = (((dp < 0) & (dq < 0)).sum(1) == 0) & (a0 <= a1)[:, 0]
    ndc = np.stack([p, q], 1)[ok]
    ndc, a0, a1 = ndc[..., :3] / ndc[..., 3:], a0[ok, 0], a1[ok, 0]
    v = np.stack([(ndc[..., 0] + 1) * 0.5 * w, (1 - ndc[..., 1]) * 0.5 * h], -1)
    v = np.floor(np.maximum(v, 0.0)).astype(np.int64)
    d = v[:, 1] - v[:, 0]
    n = np.abs(d).max(1)
    line, k = _expand(n)
    t = k / n[line]
    at = a0[line] * (1 - t) + a1[line] * t
    z = ndc[line, 0, 2] * (1 - at) + ndc[line, 1, 2] * at
    move = d[line]
    xy = v[line, 0] + np.sign(move) * (k[:, None] * np.abs(move) // n[line, None])
    ok = (xy[:, 0] < w) & (xy[:, 1] < h)
    np.minimum.at(depth, (xy[ok, 1], xy[ok, 0]), z[ok])


def exact(case, seed):
    """The depth attachments in 64 bits (colours are whole numbers)."""
    kind = case["kind"]
    if kind in ("image", "triangles") or (kind == "lines" and case["blend"]):
        return None     # no floating output
    if kind in ("batch", "serve"):
        pool, out = _pool(case, seed), []
        for w, h, k, m in _passes(case, seed):
            depth = np.ones((h, w))
            _depth_triangles(depth, _clip(*pool[k], m).reshape(-1, 3, 4))
            out.append(depth)
        return {"color": None, "depth": out[0] if len(out) == 1 else np.concatenate([d.reshape(-1) for d in out])}
    w, h = case["w"], case["h"]
    depth = np.ones((h, w))
    if kind == "lines":
        _depth_lines(depth, _clip(_lines(case, seed), None, None).reshape(-1, 2, 4))
    elif kind == "scene":
        meshes = [_mesh(seed, k, case["tris"] / 2.0 ** k, case["textured"]) for k in range(SCENE_MESHES)]
        for k, m in _objects(case, seed):
            _depth_triangles(depth, _clip(*meshes[k], m).reshape(-1, 3, 4))
    else:
        m = _camera(w, h, _rng(seed).uniform(0, 6.28))
        _depth_triangles(depth, _clip(*_mesh(seed, 0, case["tris"], case["textured"]), m).reshape(-1, 3, 4))
    return {"color": None, "depth": depth}
