"""The work that programs have this renderer do, as cases that can be timed and checked.

A case is a dict of plain values.  listed() gives the named ones, draw() another
one of the same ranges.  prepare() builds what a program holds before its frame
(a context, buffer objects, textures, display lists, captured views), run() is
one frame (or one optimisation step) through the GL 1.5 entry points, as a
program issues it: it ends with the pixels in the program's own memory.

Kinds of work:
  arrays     a lit mesh drawn with glDrawArrays from client arrays
  sphere     lit, fogged, textured spheres drawn from buffer objects
  phong      spheres lit per fragment, with exponential fog
  overdraw   many triangles, blended, stencilled and depth tested
  particles  textured quads, alpha tested and blended, from client arrays
  lists      one display list called many times under other matrices
  prims      lines and points
  pixels     a background image and sprites drawn with glDrawPixels
  batch      many contexts, recorded once and launched together
  diff       shading of captured views, forward or with its gradients
"""
import ctypes
import math

import numpy as np
import torch

import mytinygl_amd
from mytinygl_amd import ENUMS as E
from mytinygl_amd import diff as D
from mytinygl_amd import scenes as S

COLOR_DEPTH = E["GL_COLOR_BUFFER_BIT"] | E["GL_DEPTH_BUFFER_BIT"]
ALL_PLANES = COLOR_DEPTH | E["GL_STENCIL_BUFFER_BIT"]
HALF_H = 0.1          # glFrustum's half height at near = 0.1: the image is 2 units high at distance 1


def listed():
    return [
        # the smallest call: one 1,280-triangle mesh from client arrays into a
        # 640x480 window, read back.  Latency: a handful of launches and copies
        {"name": "icosphere_640x480", "kind": "arrays", "w": 640, "h": 480, "subdiv": 3, "read": "rgba"},
        # a denser mesh into an odd window, read as RGB rows
        {"name": "mesh_1001x701_rgb", "kind": "arrays", "w": 1001, "h": 701, "subdiv": 5, "read": "rgb"},
        # the ordinary frame of an interactive program: clear, one draw from
        # buffer objects with a mipmapped texture, fog and a light, present
        {"name": "textured_1080p", "kind": "sphere", "w": 1920, "h": 1080, "grid": 128, "tex": 256, "objects": 1,
         "chain": False, "read": "present"},
        # a scene of several such objects, overlapping in depth
        {"name": "textured_scene_1080p", "kind": "sphere", "w": 1920, "h": 1080, "grid": 96, "tex": 512,
         "objects": 10, "chain": False, "read": "rgba"},
        # per-fragment lighting (specular, a spot light) and exponential fog
        {"name": "phong_fog_1080p", "kind": "phong", "w": 1920, "h": 1080, "grid": 96, "read": "present"},
        # the largest: 200,000 triangles and about 100 million fragments at 4K
        {"name": "overdraw_4k", "kind": "overdraw", "w": 3840, "h": 2160, "tris": 200_000, "log_area": 4.0,
         "stencil": True, "read": "present"},
        # smoke, foliage, glass: textured quads blended over each other
        {"name": "particles_720p", "kind": "particles", "w": 1280, "h": 720, "quads": 6_000, "size": 64, "tex": 128,
         "read": "rgba"},
        # a scene of many small objects, each its own draw
        {"name": "lists_1080p", "kind": "lists", "w": 1920, "h": 1080, "copies": 64, "subdiv": 3, "read": "present"},
        # wire frames, plots and point clouds
        {"name": "lines_points_1080p", "kind": "prims", "w": 1920, "h": 1080, "lines": 100_000, "points": 100_000,
         "read": "present"},
        # video frames and overlays
        {"name": "draw_pixels_1080p", "kind": "pixels", "w": 1920, "h": 1080, "format": "GL_RGBA", "sprites": 16,
         "side": 96, "read": "present"},
        # many small independent frames: environments, thumbnails, views
        {"name": "batch_96", "kind": "batch", "contexts": 96, "fb_lo": 64, "fb_hi": 512, "tri_lo": 100,
         "tri_hi": 20_000, "draws": 4},
        # fitting colours, lights and a texture to images: one step with its gradients
        {"name": "diff_step_64", "kind": "diff", "views": 64, "side": 256, "grid": 224, "tex": 1024, "grad": True},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _window(rng):
    w = _log(rng, 161, 1920)
    return w, max(121, min(1080, int(w * rng.uniform(0.45, 0.8))))


def draw(rng):
    kind = rng.choice(["arrays", "sphere", "sphere", "phong", "overdraw", "particles", "lists", "prims", "pixels",
                       "batch", "diff", "diff"])
    if kind == "batch":
        lo = _log(rng, 48, 128)
        return {"kind": kind, "contexts": _log(rng, 8, 96), "fb_lo": lo, "fb_hi": _log(rng, lo + 16, 512),
                "tri_lo": 100, "tri_hi": _log(rng, 1_000, 20_000), "draws": rng.randint(1, 4)}
    if kind == "diff":
        return {"kind": kind, "views": _log(rng, 4, 64), "side": _log(rng, 49, 256), "grid": _log(rng, 32, 224),
                "tex": 2 ** rng.randint(7, 10), "grad": rng.random() < 0.6}
    w, h = _window(rng)
    c = {"kind": kind, "w": w, "h": h, "read": rng.choice(["rgba", "rgb", "present"])}
    if kind == "arrays":
        c["subdiv"] = rng.randint(1, 5)
    elif kind == "sphere":
        c.update(grid=_log(rng, 8, 160), tex=2 ** rng.randint(5, 10), objects=_log(rng, 1, 12),
                 chain=rng.random() < 0.25)
    elif kind == "phong":
        c["grid"] = _log(rng, 8, 128)
    elif kind == "overdraw":
        c.update(tris=_log(rng, 1_000, 200_000), log_area=round(rng.uniform(2.0, 4.0), 2), stencil=rng.random() < 0.5)
        # at most about as many layers over each pixel as the 4K frame has
        mean = 10.0 ** c["log_area"] / (c["log_area"] * math.log(10.0))
        c["tris"] = max(100, min(c["tris"], int(26 * w * h / mean)))
    elif kind == "particles":
        size = _log(rng, 6, 64)
        c.update(quads=max(50, min(_log(rng, 100, 6_000), 30 * w * h // size ** 2)), size=size,
                 tex=2 ** rng.randint(4, 8))
    elif kind == "lists":
        c.update(copies=_log(rng, 4, 64), subdiv=rng.randint(1, 3))
    elif kind == "prims":
        c.update(lines=_log(rng, 500, 100_000), points=_log(rng, 500, 100_000))
    else:
        c.update(format=rng.choice(["GL_RGBA", "GL_RGB", "GL_LUMINANCE", "GL_LUMINANCE_ALPHA"]),
                 sprites=rng.randint(0, 32), side=_log(rng, 9, min(96, h - 1)))
    return c


# ---------------------------------------------------------------------------
# contexts
# ---------------------------------------------------------------------------

class Window:
    """A context, the program's frame buffer in pinned host memory, and the GL
    calls of one frame.  The context ends with the object."""

    def __init__(self, case):
        self.w, self.h, self.read = case["w"], case["h"], case["read"]
        self.g = mytinygl_amd.load()
        self.g.lib.mtgl_present.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int32]
        self.ctx = self.g.create_context(self.w, self.h)
        self.out = torch.empty((self.h, self.w, 3 if self.read == "rgb" else 4), dtype=torch.uint8, pin_memory=True)
        self.at = self.out.data_ptr()
        self.frame = None
        self.g.glPixelStorei(E["GL_PACK_ALIGNMENT"], 1)

    def present(self):
        if self.read == "present":
            if self.g.lib.mtgl_present(self.ctx, self.at, self.w * 4):
                raise RuntimeError("mtgl_present failed")
        else:
            self.g.glReadPixels(0, 0, self.w, self.h, E["GL_RGB" if self.read == "rgb" else "GL_RGBA"],
                                E["GL_UNSIGNED_BYTE"], self.at)

    def run(self):
        self.g.gl_make_current(self.ctx)
        self.frame()
        self.present()
        return self.out

    def __del__(self):
        if getattr(self, "ctx", None):
            self.g.destroy_context(self.ctx)
            self.g.release()
            self.ctx = None


def _projection(g, w, h):
    g.glViewport(0, 0, w, h)
    g.glMatrixMode(E["GL_PROJECTION"])
    g.glLoadIdentity()
    g.glFrustum(-HALF_H * w / h, HALF_H * w / h, -HALF_H, HALF_H, 0.1, 100.0)
    g.glMatrixMode(E["GL_MODELVIEW"])
    g.glLoadIdentity()


def _lit(g):
    g.glEnable(E["GL_DEPTH_TEST"])
    g.glEnable(E["GL_LIGHTING"])
    g.glEnable(E["GL_LIGHT0"])
    g.glLightfv(E["GL_LIGHT0"], E["GL_POSITION"], g.fv(1, 1, 1, 0))


def _texture(g, texels, min_filter, mag_filter="GL_LINEAR", wrap="GL_REPEAT"):
    h, w = texels.shape[:2]
    ids = np.zeros(1, np.uint32)
    g.glGenTextures(1, ids)
    g.glBindTexture(E["GL_TEXTURE_2D"], int(ids[0]))
    g.glTexImage2D(E["GL_TEXTURE_2D"], 0, E["GL_RGBA"], w, h, 0, E["GL_RGBA"], E["GL_UNSIGNED_BYTE"],
                   g.keep(np.ascontiguousarray(texels)))
    g.glTexParameteri(E["GL_TEXTURE_2D"], E["GL_TEXTURE_MIN_FILTER"], E[min_filter])
    g.glTexParameteri(E["GL_TEXTURE_2D"], E["GL_TEXTURE_MAG_FILTER"], E[mag_filter])
    g.glTexParameteri(E["GL_TEXTURE_2D"], E["GL_TEXTURE_WRAP_S"], E[wrap])
    g.glTexParameteri(E["GL_TEXTURE_2D"], E["GL_TEXTURE_WRAP_T"], E[wrap])
    g.glEnable(E["GL_TEXTURE_2D"])


def _buffers(g, verts, idx=None):
    ids = np.zeros(2, np.uint32)
    g.glGenBuffers(2, ids)
    g.glBindBuffer(E["GL_ARRAY_BUFFER"], int(ids[0]))
    g.glBufferData(E["GL_ARRAY_BUFFER"], verts.nbytes, g.keep(np.ascontiguousarray(verts)), E["GL_STATIC_DRAW"])
    if idx is not None:
        g.glBindBuffer(E["GL_ELEMENT_ARRAY_BUFFER"], int(ids[1]))
        g.glBufferData(E["GL_ELEMENT_ARRAY_BUFFER"], idx.nbytes, g.keep(np.ascontiguousarray(idx)),
                       E["GL_STATIC_DRAW"])


def _arrays(case, seed, win):
    g, rng = win.g, np.random.default_rng([seed, 1])
    pos, faces = S.icosphere(case["subdiv"])
    tri = faces.reshape(-1)
    bump = 1.0 + 0.04 * rng.standard_normal((len(pos), 1))
    vp = np.ascontiguousarray((pos * bump)[tri].astype(np.float32))
    vn = np.ascontiguousarray(pos[tri].astype(np.float32))
    vc = np.ascontiguousarray(rng.random((len(pos), 4)).astype(np.float32)[tri])
    _projection(g, case["w"], case["h"])
    _lit(g)
    g.glEnable(E["GL_COLOR_MATERIAL"])
    g.glColorMaterial(E["GL_FRONT_AND_BACK"], E["GL_AMBIENT_AND_DIFFUSE"])
    g.glTranslatef(0.0, 0.0, -2.2)
    g.glRotatef(float(rng.uniform(0, 360)), 0.2, 1.0, 0.1)
    for a in ("GL_VERTEX_ARRAY", "GL_NORMAL_ARRAY", "GL_COLOR_ARRAY"):
        g.glEnableClientState(E[a])
    g.glVertexPointer(3, E["GL_FLOAT"], 0, g.keep(vp))
    g.glNormalPointer(E["GL_FLOAT"], 0, g.keep(vn))
    g.glColorPointer(4, E["GL_FLOAT"], 0, g.keep(vc))
    n = len(tri)

    def frame():
        g.glClear(COLOR_DEPTH)
        g.glDrawArrays(E["GL_TRIANGLES"], 0, n)
    return frame


def _sphere_places(objects, rng):
    """(x, y, distance, yaw) of each object; one object fills the image."""
    if objects == 1:
        return [(0.0, 0.0, 2.0, float(rng.uniform(0, 360)))]
    out = []
    for _ in range(objects):
        d = float(rng.uniform(2.2, 5.0))
        out.append((float(rng.uniform(-1.2, 1.2)) * d * 0.7, float(rng.uniform(-0.6, 0.6)) * d * 0.7, d,
                    float(rng.uniform(0, 360))))
    return out


def _sphere(case, seed, win):
    g, rng = win.g, np.random.default_rng([seed, 2])
    verts, idx = S.sphere_grid(case["grid"], seed + 11)
    _projection(g, case["w"], case["h"])
    _lit(g)
    g.glHint(E["GL_PERSPECTIVE_CORRECTION_HINT"], E["GL_NICEST"])
    g.glEnable(E["GL_FOG"])
    g.glFogi(E["GL_FOG_MODE"], E["GL_LINEAR"])
    g.glFogf(E["GL_FOG_START"], 1.0)
    g.glFogf(E["GL_FOG_END"], 3.0 if case["objects"] == 1 else 8.0)
    if case["chain"]:
        g.texture_lod_mode(win.ctx, 1)
    _texture(g, S.value_noise_rgba(case["tex"], seed + 12), "GL_LINEAR_MIPMAP_LINEAR")
    _buffers(g, verts, idx)
    for a in ("GL_VERTEX_ARRAY", "GL_NORMAL_ARRAY", "GL_TEXTURE_COORD_ARRAY"):
        g.glEnableClientState(E[a])
    g.glVertexPointer(3, E["GL_FLOAT"], 32, 0)
    g.glNormalPointer(E["GL_FLOAT"], 32, 12)
    g.glTexCoordPointer(2, E["GL_FLOAT"], 32, 24)
    n = len(idx)
    places = _sphere_places(case["objects"], rng)

    def frame():
        g.glClear(COLOR_DEPTH)
        for x, y, d, yaw in places:
            g.glLoadIdentity()
            g.glTranslatef(x, y, -d)
            g.glRotatef(yaw, 0.1, 1.0, 0.2)
            g.glDrawElements(E["GL_TRIANGLES"], n, E["GL_UNSIGNED_INT"], 0)
    return frame


def _phong(case, seed, win):
    g, rng = win.g, np.random.default_rng([seed, 3])
    n = S.setup_libm_spheres(g, case["w"], case["h"], seed + 21, case["grid"])
    kd = rng.uniform(0.3, 0.9, 3)
    g.glMaterialfv(E["GL_FRONT_AND_BACK"], E["GL_DIFFUSE"], g.fv(float(kd[0]), float(kd[1]), float(kd[2]), 1.0))

    def frame():
        g.glClear(COLOR_DEPTH)
        S.draw_libm_spheres(g, n)
    return frame


def _overdraw(case, seed, win):
    g = win.g
    w, h = case["w"], case["h"]
    pos, col = S.overdraw_geometry(w, h, case["tris"], seed + 31, case["log_area"])
    g.glViewport(0, 0, w, h)
    g.glMatrixMode(E["GL_PROJECTION"])
    g.glLoadIdentity()
    g.glOrtho(0.0, float(w), 0.0, float(h), 0.1, 100.0)
    g.glMatrixMode(E["GL_MODELVIEW"])
    g.glLoadIdentity()
    g.glEnable(E["GL_CULL_FACE"])
    g.glEnable(E["GL_BLEND"])
    g.glBlendFunc(E["GL_SRC_ALPHA"], E["GL_ONE_MINUS_SRC_ALPHA"])
    g.glEnable(E["GL_DEPTH_TEST"])
    if case["stencil"]:
        g.glEnable(E["GL_STENCIL_TEST"])
        g.glStencilFunc(E["GL_GREATER"], 8, 0xFF)
        g.glStencilOp(E["GL_KEEP"], E["GL_KEEP"], E["GL_INCR"])
    _buffers(g, np.concatenate([pos, col], 1).astype(np.float32))
    g.glEnableClientState(E["GL_VERTEX_ARRAY"])
    g.glEnableClientState(E["GL_COLOR_ARRAY"])
    g.glVertexPointer(3, E["GL_FLOAT"], 28, 0)
    g.glColorPointer(4, E["GL_FLOAT"], 28, 12)
    n = len(pos)

    def frame():
        g.glClear(ALL_PLANES)
        g.glDrawArrays(E["GL_TRIANGLES"], 0, n)
    return frame


def _particles(case, seed, win):
    g, rng = win.g, np.random.default_rng([seed, 4])
    w, h, nq = case["w"], case["h"], case["quads"]
    tex = S.value_noise_rgba(case["tex"], seed + 41, octaves=3, lattice=4)
    c = (np.arange(case["tex"]) + 0.5) / case["tex"] * 2 - 1        # alpha falls off to the quad's edge
    fall = np.clip(1.2 - np.sqrt(c[:, None] ** 2 + c[None, :] ** 2), 0, 1)
    tex[..., 3] = (tex[..., 3] * fall).astype(np.uint8)
    side = case["size"] * rng.uniform(0.4, 1.6, nq)
    ang = rng.uniform(0, 2 * np.pi, nq)[:, None] + np.array([0.25, 0.75, 1.25, 1.75]) * np.pi
    x = rng.uniform(0, w, nq)[:, None] + side[:, None] * 0.5 ** 0.5 * np.cos(ang)
    y = rng.uniform(0, h, nq)[:, None] + side[:, None] * 0.5 ** 0.5 * np.sin(ang)
    z = np.sort(rng.uniform(-90, -1, nq))[:, None].repeat(4, 1)      # back to front
    pos = np.ascontiguousarray(np.stack([x, y, z], -1).reshape(-1, 3).astype(np.float32))
    uv = np.ascontiguousarray(np.tile(np.array([[1, 1], [0, 1], [0, 0], [1, 0]], np.float32), (nq, 1)))
    col = np.ascontiguousarray(np.repeat(rng.random((nq, 4)).astype(np.float32), 4, 0))
    g.glViewport(0, 0, w, h)
    g.glMatrixMode(E["GL_PROJECTION"])
    g.glLoadIdentity()
    g.glOrtho(0.0, float(w), 0.0, float(h), 0.1, 100.0)
    g.glMatrixMode(E["GL_MODELVIEW"])
    g.glLoadIdentity()
    _texture(g, tex, "GL_LINEAR", wrap="GL_CLAMP")
    g.glEnable(E["GL_DEPTH_TEST"])
    g.glDepthMask(0)
    g.glEnable(E["GL_BLEND"])
    g.glBlendFunc(E["GL_SRC_ALPHA"], E["GL_ONE_MINUS_SRC_ALPHA"])
    g.glEnable(E["GL_ALPHA_TEST"])
    g.glAlphaFunc(E["GL_GREATER"], 0.02)
    for a in ("GL_VERTEX_ARRAY", "GL_TEXTURE_COORD_ARRAY", "GL_COLOR_ARRAY"):
        g.glEnableClientState(E[a])
    g.glVertexPointer(3, E["GL_FLOAT"], 0, g.keep(pos))
    g.glTexCoordPointer(2, E["GL_FLOAT"], 0, g.keep(uv))
    g.glColorPointer(4, E["GL_FLOAT"], 0, g.keep(col))

    def frame():
        g.glDepthMask(1)
        g.glClear(COLOR_DEPTH)
        g.glDepthMask(0)
        g.glDrawArrays(E["GL_QUADS"], 0, 4 * nq)
    return frame


def _lists(case, seed, win):
    g, rng = win.g, np.random.default_rng([seed, 5])
    pos, faces = S.icosphere(case["subdiv"])
    col = rng.random((len(pos), 4))
    _projection(g, case["w"], case["h"])
    g.glTranslatef(0.0, 0.0, -12.0)
    _lit(g)
    g.glEnable(E["GL_COLOR_MATERIAL"])
    lid = g.glGenLists(1)
    g.glNewList(lid, E["GL_COMPILE"])
    g.glBegin(E["GL_TRIANGLES"])
    for i in faces.reshape(-1).tolist():
        g.glColor4f(*col[i].tolist())
        g.glNormal3f(*pos[i].tolist())
        g.glVertex3f(*pos[i].tolist())
    g.glEnd()
    g.glEndList()
    copies = case["copies"]
    side = int(math.ceil(math.sqrt(copies)))
    yaw = rng.uniform(0, 360, copies).tolist()

    def frame():
        g.glClear(COLOR_DEPTH)
        for k in range(copies):
            g.glPushMatrix()
            g.glTranslatef(2.2 * (k % side - side / 2 + 0.5), 1.4 * (k // side - side / 2 + 0.5), 0.0)
            g.glScalef(0.6, 0.6, 0.6)
            g.glRotatef(yaw[k], 0.0, 1.0, 0.0)
            g.glCallList(lid)
            g.glPopMatrix()
    return frame


def _prims(case, seed, win):
    g = win.g
    st = S.setup_lines_points(g, case["w"], case["h"], seed + 51, case["lines"], case["points"])

    def frame():
        g.glClear(COLOR_DEPTH)
        S.draw_lines_points(g, st)
    return frame


_BPP = {"GL_RGBA": 4, "GL_RGB": 3, "GL_LUMINANCE": 1, "GL_LUMINANCE_ALPHA": 2}


def _pixels(case, seed, win):
    g, rng = win.g, np.random.default_rng([seed, 6])
    w, h, side = case["w"], case["h"], case["side"]
    back = g.keep(rng.integers(0, 256, w * h * _BPP[case["format"]], dtype=np.uint8))
    sprites = []
    for _ in range(case["sprites"]):
        img = g.keep(rng.integers(0, 256, side * side * 4, dtype=np.uint8))
        sprites.append((int(rng.integers(0, max(1, w - side))), int(rng.integers(0, max(1, h - side))), img))
    g.glViewport(0, 0, w, h)
    g.glMatrixMode(E["GL_PROJECTION"])
    g.glLoadIdentity()
    g.glOrtho(0.0, float(w), 0.0, float(h), -1.0, 1.0)
    g.glMatrixMode(E["GL_MODELVIEW"])
    g.glLoadIdentity()
    g.glEnable(E["GL_DEPTH_TEST"])
    g.glDepthFunc(E["GL_LEQUAL"])
    g.glBlendFunc(E["GL_SRC_ALPHA"], E["GL_ONE_MINUS_SRC_ALPHA"])
    fmt = E[case["format"]]

    def frame():
        g.glClear(COLOR_DEPTH)
        g.glDisable(E["GL_BLEND"])
        g.glRasterPos2i(0, 0)
        g.glDrawPixels(w, h, fmt, E["GL_UNSIGNED_BYTE"], back)
        g.glEnable(E["GL_BLEND"])
        for x, y, img in sprites:
            g.glRasterPos2i(x, y)
            g.glDrawPixels(side, side, E["GL_RGBA"], E["GL_UNSIGNED_BYTE"], img)
    return frame


_FRAMES = {"arrays": _arrays, "sphere": _sphere, "phong": _phong, "overdraw": _overdraw, "particles": _particles,
           "lists": _lists, "prims": _prims, "pixels": _pixels}


class Batch:
    """Many contexts, one frame of each recorded into a batch; a pass launches
    it and reads every context's image into one host buffer."""

    def __init__(self, case, seed):
        self.g = mytinygl_amd.load()
        # the sizes belong to the case, what is in the scenes to the seed
        specs = S.batch_specs(case["contexts"], S.SEED_BASE + 5, (case["fb_lo"], case["fb_hi"]),
                              (case["tri_lo"], case["tri_hi"]), (64, 256))
        rng = np.random.default_rng([seed, 8])
        for sp in specs:
            sp.update(seed=int(rng.integers(1 << 30)), yaw=float(rng.uniform(0, 360)),
                      clear=[float(c) for c in rng.random(3)])
        draws = case["draws"]

        def frame(g, n):
            g.glClear(COLOR_DEPTH)
            for k in range(draws):
                g.glPushMatrix()
                g.glTranslatef(0.9 * (k % 2) - 0.45 * (draws > 1), 0.9 * (k // 2) - 0.45 * (draws > 2), -0.6 * k)
                g.glDrawElements(E["GL_TRIANGLES"], n, E["GL_UNSIGNED_INT"], 0)
                g.glPopMatrix()

        items = [(sp["w"], sp["h"], (lambda g, sp=sp: S.setup_batch_scene(g, sp)), frame) for sp in specs]
        self.set = S.BatchRun(self.g, items)
        self.batch = self.set.record(autotune=False)
        sizes = [sp["w"] * sp["h"] * 4 for sp in specs]
        self.out = torch.empty(sum(sizes), dtype=torch.uint8, pin_memory=True)
        at, self.images = self.out.data_ptr(), []
        for ctx, sp, n in zip(self.set.ctxs, specs, sizes):
            self.images.append((ctx, sp["w"], sp["h"], at))
            at += n

    def run(self):
        g = self.g
        self.batch.launch()
        for ctx, w, h, at in self.images:
            g.gl_make_current(ctx)
            g.glReadPixels(0, 0, w, h, E["GL_RGBA"], E["GL_UNSIGNED_BYTE"], at)
        return self.out

    def __del__(self):
        if getattr(self, "set", None) is not None:
            self.set.close()
            self.set = None


class Diff:
    """Captured views, the parameters and the target images of a fit."""

    def __init__(self, case, seed):
        self.params = D.diff_params(case["grid"], case["tex"], case["views"], seed + 71)
        # moved a little from the views' own look-at points: other pixels for other seeds
        rng = np.random.default_rng([seed, 7])
        self.params["eyes"] = self.params["eyes"] * rng.uniform(0.9, 1.2, (case["views"], 1))
        self.g = mytinygl_amd.load()
        self.views = D.DiffViews(self.g, self.params, case["side"], case["side"])
        self.leaf = [torch.from_numpy(self.params[k]).cuda().requires_grad_(case["grad"])
                     for k in ("vcol", "light_rgb", "tex")]
        self.target = None
        if case["grad"]:
            moved = D.perturbed(self.params, seed + 72)
            with torch.no_grad():
                self.target = D.render(*(torch.from_numpy(moved[k]).cuda() for k in ("vcol", "light_rgb", "tex")),
                                       self.views)

    def run(self):
        image = D.render(*self.leaf, self.views)
        if self.target is None:
            return {"image": image}
        for p in self.leaf:
            p.grad = None
        ((image - self.target) ** 2).sum().backward()
        return {"image": image.detach(), "vcol": self.leaf[0].grad, "light_rgb": self.leaf[1].grad,
                "tex": self.leaf[2].grad}

    def __del__(self):
        if getattr(self, "views", None) is not None:
            self.views.close()
            self.views = None


def prepare(case, seed):
    if case["kind"] == "batch":
        return Batch(case, seed)
    if case["kind"] == "diff":
        return Diff(case, seed)
    win = Window(case)
    win.g.glClearColor(0.05, 0.1, 0.15, 1.0)
    win.frame = _FRAMES[case["kind"]](case, seed, win)
    return win


def run(state):
    return state.run()


# ---------------------------------------------------------------------------
# work and correctness
# ---------------------------------------------------------------------------

VERTEX_FLOPS = 150      # transform, one light, divide and mapping of a vertex
FRAGMENT_FLOPS = 25     # three edges, depth
SHADE_FLOPS = 60        # colour, texture coordinates, taps


def _disk(h, d, radius=1.0):
    """Pixels of a sphere of that radius at distance d in an image h high."""
    r = h / 2.0 * radius / math.sqrt(max(d * d - radius * radius, 1e-3))
    return math.pi * r * r


def work(case):
    kind = case["kind"]
    if kind == "diff":
        v, px = case["views"], case["views"] * case["side"] ** 2
        nv, tx = (case["grid"] + 1) ** 2, case["tex"] ** 2
        covered = v * min(case["side"] ** 2, _disk(case["side"], 3.1))
        read = v * nv * 24 + nv * 16 + tx * 16 + px * 40 + 6 * case["grid"] ** 2 * 4 * v
        if not case["grad"]:
            return {"bytes": read + px * 16, "flops": v * nv * 120 + covered * 60}
        # forward, loss and adjoint: the images and their targets, the gradients
        return {"bytes": 2 * read + px * 16 * 4 + nv * 16 + tx * 16, "flops": v * nv * 400 + covered * 240}
    if kind == "batch":
        # sides and triangle counts are spread over their logarithm
        lo, hi = case["fb_lo"], case["fb_hi"]
        px = case["contexts"] * ((hi * hi - lo * lo) / (2 * math.log(hi / lo)))
        tri = case["contexts"] * (case["tri_hi"] - case["tri_lo"]) / math.log(case["tri_hi"] / case["tri_lo"])
        frags = 2 * px * 0.35 * case["draws"]
        return {"bytes": tri * (16 + 12) + px * 12,
                "flops": case["draws"] * tri * 0.5 * VERTEX_FLOPS + frags * FRAGMENT_FLOPS + frags / 2 * SHADE_FLOPS}
    px = case["w"] * case["h"]
    planes = 12             # colour and depth written, colour read out
    verts = frags = shaded = inputs = 0
    if kind == "arrays":
        verts = 60 * 4 ** case["subdiv"]
        inputs = verts * 40
        shaded = min(px, _disk(case["h"], 2.2))
        frags = 2 * shaded
    elif kind == "sphere":
        n = case["objects"]
        verts = n * (case["grid"] + 1) ** 2
        inputs = (case["grid"] + 1) ** 2 * 32 + 24 * case["grid"] ** 2 + case["tex"] ** 2 * 4
        shaded = n * min(px, _disk(case["h"], 2.0 if n == 1 else 3.4))
        frags = 2 * shaded
    elif kind == "phong":
        verts = 2 * (case["grid"] + 1) ** 2
        inputs = (case["grid"] + 1) ** 2 * 24 + 24 * case["grid"] ** 2
        shaded = _disk(case["h"], 2.6) + _disk(case["h"], 3.0)
        frags = 2 * shaded
        shaded *= 3
    elif kind == "overdraw":
        verts = 3 * case["tris"]
        inputs = verts * 28
        frags = case["tris"] / 2 * 10.0 ** case["log_area"] / (case["log_area"] * math.log(10.0))
        shaded = frags / 4 if case["stencil"] else frags / 3
        planes += 1
    elif kind == "particles":
        verts = 4 * case["quads"]
        inputs = verts * 36 + case["tex"] ** 2 * 4
        frags = shaded = case["quads"] * 1.12 * case["size"] ** 2 * 0.95
    elif kind == "lists":
        verts = case["copies"] * 60 * 4 ** case["subdiv"]
        inputs = 60 * 4 ** case["subdiv"] * 52
        shaded = case["copies"] * _disk(case["h"], 12.0, 0.6)
        frags = 2 * shaded
    elif kind == "prims":
        verts = 2 * case["lines"] + case["points"]
        inputs = verts * 28
        frags = shaded = case["points"] * 9 + case["lines"] * 2 * 0.02 * case["h"]
    else:
        inputs = px * _BPP[case["format"]] + case["sprites"] * case["side"] ** 2 * 4
        shaded = px + case["sprites"] * case["side"] ** 2
    return {"bytes": inputs + px * planes,
            "flops": verts * VERTEX_FLOPS + frags * FRAGMENT_FLOPS + shaded * SHADE_FLOPS}


def tolerance(case):
    # rendered pixels are bytes whose every step is defined: they stay the same
    if case["kind"] != "diff":
        return "exact"
    # fp32 shading; gradients are fp32 sums over the pixels and views in no fixed order
    return {"rel": 4e-6, "max": 1e-4}


def exact(case, seed):
    """The diff kind in 64 bits: shading of the captured visibility (the
    G-buffer a fit holds), and its gradients by autograd.  None for images,
    which are bytes."""
    if case["kind"] != "diff":
        return None
    state = Diff(case, seed)
    P = state.params
    dev, f64 = "cuda", torch.float64
    leaf = [torch.from_numpy(P[k]).to(dev, f64).requires_grad_(case["grad"]) for k in ("vcol", "light_rgb", "tex")]
    vcol, light, tex = leaf
    idx = torch.from_numpy(P["idx"].astype(np.int64)).to(dev).reshape(-1, 3)
    normal = P["verts"][:, 3:6].astype(np.float64)
    L = P["light_dir"].astype(np.float64)
    L /= np.linalg.norm(L, axis=1, keepdims=True)
    images = []
    for v in range(case["views"]):
        mv = D.look_at(P["eyes"][v]).astype(np.float64).reshape(4, 4).T
        n = normal @ np.linalg.inv(mv[:3, :3])
        n /= np.linalg.norm(n, axis=1, keepdims=True)
        ndl = torch.from_numpy(np.maximum(n @ L.T, 0.0)).to(dev)
        gb = state.views.gbuffer(v).reshape(-1)
        at = np.nonzero(gb["tri"] >= 0)[0]
        c = gb[at]
        k = vcol.clamp(0.0, 1.0)
        rgb = k[:, :3] * (0.2 + ndl @ light)                      # the model's ambient light, then each light
        alpha = k[:, 3:] * (1.0 + len(L) + ndl.sum(1, keepdim=True))
        lit = torch.cat([rgb, alpha], 1).clamp(0.0, 1.0)
        b = torch.from_numpy(c["b"].astype(np.float64)).to(dev)
        t = torch.from_numpy(c["texel"].astype(np.int64)).to(dev)
        fx = torch.from_numpy(c["fx"].astype(np.float64)).to(dev)[:, None]
        fy = torch.from_numpy(c["fy"].astype(np.float64)).to(dev)[:, None]
        el = idx[torch.from_numpy(c["tri"].astype(np.int64)).to(dev)]
        col = (lit[el] * b[..., None]).sum(1)
        q = tex.reshape(-1, 4)
        top = q[t[:, 0]] * (1 - fx) + q[t[:, 1]] * fx
        bot = q[t[:, 2]] * (1 - fx) + q[t[:, 3]] * fx
        img = torch.zeros((case["side"] ** 2, 4), dtype=f64, device=dev)
        bg = np.nonzero(gb["tri"] < 0)[0]
        byte = (gb["texel"][bg, 0][:, None] >> np.array([0, 8, 16, 24], np.uint32)) & 0xFF
        img[torch.from_numpy(bg).to(dev)] = torch.from_numpy(byte / 255.0).to(dev)
        covered = torch.from_numpy(at).to(dev)
        image = img.index_put((covered,), (col * (top * (1 - fy) + bot * fy)).clamp(0.0, 1.0))
        image = image.reshape(case["side"], case["side"], 4)
        if case["grad"]:
            ((image - state.target[v].to(f64)) ** 2).sum().backward()
        images.append(image.detach())
    out = {"image": torch.stack(images)}
    if case["grad"]:
        out.update(vcol=leaf[0].grad, light_rgb=leaf[1].grad, tex=leaf[2].grad)
    return out
