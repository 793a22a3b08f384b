"""The rendering work whose speed is tracked: what a program that uses this
package has it do, forward and backward, through its public functions.

`listed()` holds the named cases, `draw(rng)` gives further ones of the same
ranges.  A case is a dict with a `kind`:

  fit     the inverse-rendering samples' step on a small mesh: rasterize,
          interpolate, (pie: antialias), MSE, gradients
  chain   the textured-mesh step: rasterize with screen derivatives,
          interpolate UVs, trilinear texture, antialias, MSE, gradients to
          pos, the UVs and the texture
  peel    depth-peeled layers of a dense mesh, each interpolated, gradients
          to pos and the attributes from given cotangents
  range   many meshes in one vertex buffer (ranges), a cube-map lookup with
          mip levels and a per-pixel bias, all gradients
  raster  rasterize with screen derivatives, and its gradient
  interp  interpolate alone (a G-buffer's attribute set), all gradients
  tex     texture alone (filters, boundaries, channel counts), all gradients
  cube    bilinear cube-map lookup (an environment map), texture gradient
  aa      antialias alone, gradients to colour and pos

Everything is float32 with int32 indices, the only types the package takes.
`exact` is the same work in float64 with plain torch.
"""
import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "mlx-swift-diffrast_amd"))

DEV = "cuda" if torch.cuda.is_available() else "cpu"


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------

def listed():
    return [
        # the colour-fit sample: one triangle, one small image; every call is
        # a few microseconds of GPU work, so launches and host time count
        dict(name="fit triangle 1x256^2", kind="fit", mesh="triangle", n=1, h=256, w=256),
        # the mesh-fit sample's layout on a small batch, with antialias
        dict(name="fit pie 4x512^2", kind="fit", mesh="pie", n=4, h=512, w=512),
        # one view of a light mesh, as an interactive fit renders it
        dict(name="chain 1x512^2", kind="chain", n=1, h=512, w=512, level=5, tex=512),
        # the benchmark's batch: 80k triangles, eight views, 1024^2 texture
        dict(name="chain 8x1024^2", kind="chain", n=8, h=1024, w=1024, level=6, tex=1024),
        # the dense mesh: 1.3M triangles, four peeled layers, sixteen views
        dict(name="peel 16x2048^2", kind="peel", n=16, h=2048, w=2048, level=8, layers=4),
        # thousands of independent small meshes in one call
        dict(name="range 4096x256^2", kind="range", n=4096, h=256, w=256, tris=512, size=512),
        # one UHD frame (a ragged last tile row, more tiles than the batch
        # cases have per image) of a 330k-triangle mesh
        dict(name="raster 1x2160x3840", kind="raster", n=1, h=2160, w=3840, level=7),
        # a deferred shader's G-buffer: uv, normal and colour, with screen
        # derivatives for the uv only
        dict(name="interp 4x720x1280x8", kind="interp", n=4, h=720, w=1280, level=6, a=8,
             diff="0,1"),
        # an RGB photo texture, tiled, bilinear (odd sizes)
        dict(name="tex linear 4x1000^2x3", kind="tex", n=4, h=1000, w=1000, th=600, tw=1000, c=3,
             filter="linear", boundary="wrap", bias="none"),
        # a learned feature texture (neural texture), trilinear
        dict(name="tex mip 2x768^2x16", kind="tex", n=2, h=768, w=768, th=512, tw=512, c=16,
             filter="linear-mipmap-linear", boundary="clamp", bias="none"),
        # an environment map behind and on a reflective object
        dict(name="cube 4x800^2x3", kind="cube", n=4, h=800, w=800, size=256, c=3),
        # silhouettes and shaded RGB of a medium mesh
        dict(name="aa 8x512^2x3", kind="aa", n=8, h=512, w=512, level=5, c=3),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _image(rng, lo, hi, pixels):
    """n, h, w: sides of lo..hi (odd ones too, not always square), a batch
    that keeps n * h * w within `pixels`."""
    h = _log_int(rng, lo, hi)
    w = h if rng.random() < 0.5 else max(lo, min(hi, int(h * rng.uniform(0.5, 2.0))))
    n = _log_int(rng, 1, max(1, min(16, pixels // (h * w))))
    return dict(n=n, h=h, w=w)


def draw(rng):
    kind = rng.choice(["fit", "chain", "peel", "range", "raster", "interp", "tex", "tex", "cube",
                       "aa"])
    if kind == "fit":
        return dict(kind=kind, mesh=rng.choice(["triangle", "pie"]), **_image(rng, 64, 512, 1 << 20))
    if kind == "chain":
        return dict(kind=kind, level=rng.randint(3, 6), tex=rng.choice([256, 512, 768, 1024]),
                    **_image(rng, 128, 1024, 8 << 20))
    if kind == "peel":
        return dict(kind=kind, level=rng.randint(5, 8), layers=rng.randint(2, 4),
                    **_image(rng, 256, 2048, 16 << 20))
    if kind == "range":
        return dict(kind=kind, n=_log_int(rng, 16, 1024), h=rng.randint(60, 256),
                    w=rng.randint(60, 256), tris=_log_int(rng, 16, 512),
                    size=rng.choice([64, 128, 256, 512]))
    if kind == "raster":
        return dict(kind=kind, level=rng.randint(2, 7), **_image(rng, 200, 3840, 16 << 20))
    if kind == "interp":
        a = rng.randint(1, 16)
        diff = rng.choice(["", "all", "0", ",".join(str(i) for i in range(min(a, 2)))])
        return dict(kind=kind, level=rng.randint(4, 6), a=a, diff=diff,
                    **_image(rng, 200, 1280, 4 << 20))
    if kind == "tex":
        mip = rng.random() < 0.5
        filt = rng.choice(["linear-mipmap-linear", "linear-mipmap-nearest"]) if mip else \
            rng.choice(["linear", "linear", "nearest"])
        th = rng.choice([128, 256, 512, 768, 1024]) if mip else rng.randint(100, 1024)
        tw = rng.choice([128, 256, 512, 768, 1024]) if mip else rng.randint(100, 1024)
        return dict(kind=kind, th=th, tw=tw, c=rng.choice([1, 2, 3, 3, 4, 4, 5, 6, 8, 12, 16]),
                    filter=filt, boundary=rng.choice(["wrap", "clamp", "zero"]),
                    bias=rng.choice(["none", "map", "scalar"]) if mip else "none",
                    **_image(rng, 200, 1280, 4 << 20))
    if kind == "cube":
        return dict(kind=kind, size=_log_int(rng, 32, 512), c=rng.choice([1, 3, 3, 4, 8]),
                    **_image(rng, 200, 1024, 4 << 20))
    return dict(kind="aa", level=rng.randint(3, 6), c=rng.choice([1, 3, 3, 4, 4, 8]),
                **_image(rng, 128, 1024, 4 << 20))


# ---------------------------------------------------------------------------
# scenes
# ---------------------------------------------------------------------------

@functools.lru_cache(maxsize=None)
def icosphere(level):
    """Unit icosphere on the device: vertices [V,3] float64, faces [T,3]
    int64 (10 * 4^level + 2 vertices, 20 * 4^level faces)."""
    t = (1.0 + 5.0 ** 0.5) / 2.0
    v = torch.tensor([[-1, t, 0], [1, t, 0], [-1, -t, 0], [1, -t, 0], [0, -1, t], [0, 1, t],
                      [0, -1, -t], [0, 1, -t], [t, 0, -1], [t, 0, 1], [-t, 0, -1], [-t, 0, 1]],
                     dtype=torch.float64, device=DEV)
    f = torch.tensor([[0, 11, 5], [0, 5, 1], [0, 1, 7], [0, 7, 10], [0, 10, 11], [1, 5, 9],
                      [5, 11, 4], [11, 10, 2], [10, 7, 6], [7, 1, 8], [3, 9, 4], [3, 4, 2],
                      [3, 2, 6], [3, 6, 8], [3, 8, 9], [4, 9, 5], [2, 4, 11], [6, 2, 10],
                      [8, 6, 7], [9, 8, 1]], device=DEV)
    v = v / v.norm(dim=1, keepdim=True)
    for _ in range(level):
        e = torch.cat([f[:, [0, 1]], f[:, [1, 2]], f[:, [2, 0]]]).sort(dim=1).values
        uk, inv = torch.unique(e[:, 0] * (1 << 32) + e[:, 1], return_inverse=True)
        mid = v[uk >> 32] + v[uk & 0xFFFFFFFF]
        base, F = v.shape[0], f.shape[0]
        v = torch.cat([v, mid / mid.norm(dim=1, keepdim=True)])
        m01, m12, m20 = base + inv[:F], base + inv[F:2 * F], base + inv[2 * F:]
        f = torch.cat([torch.stack([f[:, 0], m01, m20], 1), torch.stack([f[:, 1], m12, m01], 1),
                       torch.stack([f[:, 2], m20, m12], 1), torch.stack([m01, m12, m20], 1)])
    return v, f


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _rotations(n, seed):
    q = np.random.default_rng(seed).normal(size=(n, 4))
    w, x, y, z = (q / np.linalg.norm(q, axis=1, keepdims=True)).T
    R = np.stack([1 - 2 * (y * y + z * z), 2 * (x * y - z * w), 2 * (x * z + y * w),
                  2 * (x * y + z * w), 1 - 2 * (x * x + z * z), 2 * (y * z - x * w),
                  2 * (x * z - y * w), 2 * (y * z + x * w), 1 - 2 * (x * x + y * y)], 1)
    return torch.as_tensor(R.reshape(n, 3, 3), device=DEV)


def _project(v, R, dist=3.0, fov=45.0, near=1.0, far=10.0):
    """Clip-space pos [N,V,4] of a unit-sized mesh seen from `dist`."""
    f = 1.0 / math.tan(math.radians(fov) / 2)
    cam = v @ R.transpose(1, 2)
    x, y, z = cam[..., 0], cam[..., 1], cam[..., 2] - dist
    a, b = (far + near) / (near - far), 2 * far * near / (near - far)
    return torch.stack([f * x, f * y, a * z + b, -z], -1).float().contiguous()


def _displaced(v, seed):
    rng = np.random.default_rng(seed)
    k = torch.as_tensor(rng.normal(size=(8, 3)) * 3.0, device=DEV)
    ph = torch.as_tensor(rng.uniform(0, 2 * np.pi, size=8), device=DEV)
    return v * (1.0 + 0.1 * torch.sin(v @ k.T + ph).mean(dim=1))[:, None]


def _spherical_uv(m):
    return torch.stack([0.5 + torch.atan2(m[..., 2], m[..., 0]) / (2 * math.pi),
                        0.5 - torch.asin(m[..., 1].clamp(-1, 1)) / math.pi], -1)


def _noise(shape, gen):
    """A smooth random image [n, h, w, c] in [0, 1] (three octaves)."""
    n, h, w, c = shape
    out = torch.zeros((n, c, h, w), device=DEV)
    for amp, g in ((1.0, 8), (0.5, 32), (0.25, 128)):
        grid = torch.rand((n, c, g + 1, g + 1), device=DEV, generator=gen)
        out += amp * torch.nn.functional.interpolate(grid, size=(h, w), mode="bilinear",
                                                     align_corners=True)
    return (out / 1.75).permute(0, 2, 3, 1).contiguous()


def _sphere_view(n, h, w, seed):
    """What the pixels of n images of a textured sphere see: which pixels are
    covered [n,h,w], the rotated unit normal there (an unrotated view ray
    elsewhere) and its screen derivatives, float64."""
    R = _rotations(n, seed)
    s = 2.0 / min(h, w)
    x = (torch.arange(w, device=DEV, dtype=torch.float64) + 0.5 - w / 2) * s
    y = -(torch.arange(h, device=DEV, dtype=torch.float64) + 0.5 - h / 2) * s
    x, y = (x / 0.85)[None, :].expand(h, w), (y / 0.85)[:, None].expand(h, w)
    zz = 1.0 - x * x - y * y
    cov = zz > 1e-6
    z = torch.sqrt(torch.where(cov, zz, torch.ones_like(zz)))
    nrm = torch.where(cov[..., None], torch.stack([x, y, z], -1),
                      torch.stack([x, y, -1.5 * torch.ones_like(x)], -1))
    d = s / 0.85
    one, zero = torch.ones_like(x), torch.zeros_like(x)
    dx = torch.stack([one, zero, -x / z], -1) * d
    dy = -torch.stack([zero, one, -y / z], -1) * d
    rot = lambda a: torch.einsum("nij,hwj->nhwi", R, a)  # noqa: E731
    return cov[None].expand(n, h, w), rot(nrm), rot(dx), rot(dy)


def _uv_field(case, seed):
    """uv [n,h,w,2] and uvDA [n,h,w,4] of a textured sphere; empty pixels are
    zero, as interpolate leaves them."""
    cov, m, dx, dy = _sphere_view(case["n"], case["h"], case["w"], seed)
    rep = 3.0 if case["boundary"] == "wrap" else 1.0
    uv = _spherical_uv(m / m.norm(dim=-1, keepdim=True))
    hyp = (m[..., 0] ** 2 + m[..., 2] ** 2).clamp_min(1e-9)
    du = [(m[..., 0] * d[..., 2] - m[..., 2] * d[..., 0]) / hyp / (2 * math.pi) for d in (dx, dy)]
    dv = [-d[..., 1] / torch.sqrt((1 - m[..., 1] ** 2).clamp_min(1e-9)) / math.pi for d in (dx, dy)]
    if case["boundary"] == "zero":  # a decal smaller than the surface
        uv = uv * 1.25 - 0.125
    uv = uv * rep * cov[..., None]
    da = torch.stack(du + dv, -1) * rep * cov[..., None]
    return uv.float().contiguous(), da.float().contiguous()


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _i32(t):
    return t.to(torch.int32).contiguous()


def _inputs(case, seed):
    """The case's input tensors by name (leaves that take gradients are
    named in _LEAVES)."""
    k, g = case["kind"], _gen(seed)
    rand = lambda *s: torch.rand(s, device=DEV, generator=g)  # noqa: E731
    randn = lambda *s: torch.randn(s, device=DEV, generator=g)  # noqa: E731
    n, h, w = case["n"], case["h"], case["w"]
    if k == "fit":
        if case["mesh"] == "triangle":  # x, y in [-0.8, 0.8], wide enough to be seen
            ang = rand(n, 1) * 6.28 + torch.tensor([0.0, 2.1, 4.2], device=DEV)
            rad = 0.5 + 0.3 * rand(n, 3)
            tri = torch.tensor([[0, 1, 2]], device=DEV)
        else:  # a centre and six ring vertices, slightly moved per image
            a = torch.arange(6, device=DEV) * (math.pi / 3)
            ang = torch.cat([torch.zeros(1, device=DEV), a]).expand(n, 7) + 0.03 * randn(n, 7)
            rad = torch.cat([torch.zeros(1, device=DEV), torch.full((6,), 0.6, device=DEV)]) + \
                0.02 * randn(n, 7)
            tri = torch.tensor([[0, i, i % 6 + 1] for i in range(1, 7)], device=DEV)
        xy = torch.stack([rad * torch.cos(ang), rad * torch.sin(ang)], -1)
        pos = torch.cat([xy, torch.zeros_like(xy[..., :1]), torch.ones_like(xy[..., :1])], -1)
        return dict(pos=pos.contiguous(), tri=_i32(tri), attr=rand(1, pos.shape[1], 3),
                    target=rand(n, h, w, 3))
    if k in ("chain", "peel", "raster", "interp", "aa"):
        v, f = icosphere(case["level"])
        shape = _displaced(v, seed) if k in ("peel", "interp", "aa") else v
        pos, tri = _project(shape, _rotations(n, seed + 1)), _i32(f)
    if k == "chain":
        tex = _noise((1, case["tex"], case["tex"], 4), g)
        return dict(pos=pos, tri=tri, attr=_spherical_uv(v).float().contiguous(), tex=tex,
                    target=rand(n, h, w, 4))
    if k == "peel":
        attr = torch.cat([v.float(), rand(v.shape[0], 3)], 1)[None].contiguous()
        return dict(pos=pos, tri=tri, attr=attr,
                    **{"g%d" % i: randn(n, h, w, 6) * 1e-3 for i in range(case["layers"])})
    if k == "range":
        t = case["tris"]
        V = n * t * 3
        pos = torch.cat([rand(V, 3) * 2 - 1, torch.ones((V, 1), device=DEV)], 1)
        ranges = torch.stack([torch.arange(n) * t, torch.full((n,), t)], 1).to(torch.int32)
        hh = 1 - 2 * (torch.arange(h, device=DEV) + 0.5) / h
        ww = 1 - 2 * (torch.arange(w, device=DEV) + 0.5) / w
        env = torch.stack([torch.ones((h, w), device=DEV), hh[:, None].expand(h, w),
                           ww[None, :].expand(h, w)], -1).contiguous()
        s = case["size"]
        return dict(pos=pos, tri=_i32(torch.arange(V, device=DEV).reshape(-1, 3)), ranges=ranges,
                    attr=randn(V, 3), cube=rand(1, 6, s, s, 3), bias=rand(n, h, w) * 2 - 1,
                    env=env, g=randn(n, h, w, 3) * 1e-3)
    if k == "raster":
        return dict(pos=pos, tri=tri, g=randn(n, h, w, 4), gdb=randn(n, h, w, 4) * 1e-2)
    if k == "interp":
        tid = cover(pos, tri, h, w)
        rast, db = bary(pos.double(), tri, tid, h, w)
        K = _n_diff(case)
        return dict(attr=randn(n, v.shape[0], case["a"]), rast=rast.float(), rast_db=db.float(),
                    tri=tri, g=randn(n, h, w, case["a"]), gda=randn(n, h, w, 2 * K))
    if k == "tex":
        uv, da = _uv_field(case, seed)
        d = dict(tex=_noise((1, case["th"], case["tw"], case["c"]), g), uv=uv,
                 g=randn(n, h, w, case["c"]))
        if "mipmap" in case["filter"]:
            d["uv_da"] = da
        if case["bias"] == "map":
            d["bias"] = rand(n, h, w) * 2 - 1
        return d
    if k == "cube":
        _, m, _, _ = _sphere_view(n, h, w, seed)
        s = case["size"]
        return dict(tex=rand(1, 6, s, s, case["c"]), uv=m.float().contiguous(),
                    g=randn(n, h, w, case["c"]))
    rast = bary(pos.double(), tri, cover(pos, tri, h, w), h, w)[0].float()
    color = torch.where(rast[..., 3:] > 0, _noise((n, h, w, case["c"]), g),
                        torch.zeros((), device=DEV)).contiguous()
    return dict(color=color, rast=rast, pos=pos, tri=tri, g=randn(n, h, w, case["c"]))


def _n_diff(case):
    d = case.get("diff", "")
    return case["a"] if d == "all" else (len(d.split(",")) if d else 0)


_LEAVES = {"fit": ["pos", "attr"], "chain": ["pos", "attr", "tex"], "peel": ["pos", "attr"],
           "range": ["pos", "attr", "cube"], "raster": ["pos"],
           "interp": ["attr", "rast", "rast_db"], "tex": ["tex", "uv", "uv_da", "bias"],
           "cube": ["tex"], "aa": ["color", "pos"]}


def _leaves(case):
    names = list(_LEAVES[case["kind"]])
    if case["kind"] == "fit" and case["mesh"] == "triangle":
        names = ["attr"]  # the colour fit moves no vertex
    if case["kind"] == "interp" and not _n_diff(case):
        names.remove("rast_db")
    return names


def prepare(case, seed):
    from diffrast import DiffRast
    d = _inputs(case, seed)
    if case["kind"] in ("fit", "chain", "aa"):  # the mesh's topology, made once
        d["topo"] = DiffRast.antialiasConstructTopologyHash(d["tri"])
    leaves = [name for name in _leaves(case) if name in d]
    for name in leaves:
        d[name].requires_grad_(True)
    d["case"], d["leaves"] = case, leaves
    return d


def run(s):
    from diffrast import DiffRast
    from diffrast.fit import mse_loss
    case = s["case"]
    k = case["kind"]
    size = (case["h"], case["w"])
    if k == "fit":
        rast, _ = DiffRast.rasterize(s["pos"], s["tri"], size, gradDB=False)
        out, _ = DiffRast.interpolate(s["attr"], rast, s["tri"])
        if case["mesh"] == "pie":
            out = DiffRast.antialias(out, rast, s["pos"], s["tri"], topologyHash=s["topo"])
        outs, grads = {"loss": mse_loss(out, s["target"]), "image": out}, None
    elif k == "chain":
        rast, db = DiffRast.rasterize(s["pos"], s["tri"], size, gradDB=True)
        uv, uv_da = DiffRast.interpolate(s["attr"], rast, s["tri"], rastDB=db, diffAttrs="all")
        col = DiffRast.texture(s["tex"], uv, uvDA=uv_da, filterMode="linear-mipmap-linear",
                               boundaryMode="clamp")
        out = DiffRast.antialias(col, rast, s["pos"], s["tri"], topologyHash=s["topo"])
        outs, grads = {"loss": mse_loss(out, s["target"]), "image": out}, None
    elif k == "peel":
        outs, prev = {}, None
        for i in range(case["layers"]):
            rast, _ = DiffRast.rasterize(s["pos"], s["tri"], size, gradDB=False, peelLayer=prev)
            outs["layer%d" % i], _ = DiffRast.interpolate(s["attr"], rast, s["tri"])
            prev = rast.detach()
        grads = [s["g%d" % i] for i in range(case["layers"])]
    elif k == "range":
        rast, db = DiffRast.rasterize(s["pos"], s["tri"], size, gradDB=True, ranges=s["ranges"])
        dirs, da = DiffRast.interpolate(s["attr"], rast, s["tri"], rastDB=db, diffAttrs="all")
        dirs = dirs + (rast[..., 3:4] == 0).float() * s["env"]  # empty pixels see the background
        outs = {"image": DiffRast.texture(s["cube"], dirs, uvDA=da,
                                          filterMode="linear-mipmap-linear", boundaryMode="cube",
                                          mipLevelBiasMap=s["bias"], dirGrad=True)}
        grads = [s["g"]]
    elif k == "raster":
        rast, db = DiffRast.rasterize(s["pos"], s["tri"], size, gradDB=True)
        outs, grads = {"rast": rast, "rast_db": db}, [s["g"], s["gdb"]]
    elif k == "interp":
        if _n_diff(case):
            diff = "all" if case["diff"] == "all" else [int(i) for i in case["diff"].split(",")]
            out, da = DiffRast.interpolate(s["attr"], s["rast"], s["tri"], rastDB=s["rast_db"],
                                           diffAttrs=diff)
            outs, grads = {"out": out, "out_da": da}, [s["g"], s["gda"]]
        else:
            outs, grads = {"out": DiffRast.interpolate(s["attr"], s["rast"], s["tri"])[0]}, [s["g"]]
    elif k in ("tex", "cube"):
        kw = dict(filterMode="linear", boundaryMode="cube") if k == "cube" else \
            dict(filterMode=case["filter"], boundaryMode=case["boundary"])
        if "uv_da" in s:
            kw.update(uvDA=s["uv_da"], mipLevelBiasMap=s.get("bias"),
                      mipLevelBias=0.5 if case["bias"] == "scalar" else 0.0)
        outs, grads = {"out": DiffRast.texture(s["tex"], s["uv"], **kw)}, [s["g"]]
    else:
        outs = {"out": DiffRast.antialias(s["color"], s["rast"], s["pos"], s["tri"],
                                          topologyHash=s["topo"])}
        grads = [s["g"]]
    # a loss is back-propagated by itself; other outputs from their cotangents
    heads = [outs["loss"]] if "loss" in outs else list(outs.values())
    got = torch.autograd.grad(heads, [s[name] for name in s["leaves"]], grads)
    outs.update(("d_" + name, v) for name, v in zip(s["leaves"], got))
    return outs


# ---------------------------------------------------------------------------
# work and tolerances
# ---------------------------------------------------------------------------

def work(case):
    """Bytes: every op of the case reads its inputs and writes its outputs
    once, forward and backward (float32 pixels, the mesh and the textures
    beside them).  Flops: the arithmetic of the pixels' formulas, roughly."""
    k = case["kind"]
    P = case["n"] * case["h"] * case["w"]
    mesh = 0
    if "level" in case:
        V, T = 10 * 4 ** case["level"] + 2, 20 * 4 ** case["level"]
        mesh = 2 * case["n"] * V * 16 + T * 12
    if k == "fit":
        b = {"triangle": 16 + 28 + 36 + 44, "pie": 16 + 28 + 40 + 36 + 52 + 44 + 32}[case["mesh"]]
        return {"bytes": b * P, "flops": 100.0 * P}
    if k == "chain":
        pyr = 4.0 / 3.0 * case["tex"] ** 2 * 16
        return {"bytes": (440 + 48) * P + 6 * pyr + 4 * mesh, "flops": 600.0 * P}
    if k == "peel":
        L = case["layers"]
        b = 16 * L + 16 * (L - 1) + L * 40 + L * 56 + L * 32
        return {"bytes": b * P + 2 * mesh, "flops": 200.0 * L * P}
    if k == "range":
        V = case["n"] * case["tris"] * 3
        cube = 4.0 / 3.0 * 6 * case["size"] ** 2 * 12
        b = 32 + 68 + 28 + 52 + 84 + 100 + 48
        return {"bytes": b * P + 56 * V + 3 * cube, "flops": 900.0 * P}
    if k == "raster":
        return {"bytes": (32 + 48) * P + 2 * mesh, "flops": 250.0 * P}
    if k == "interp":
        a, K = case["a"], _n_diff(case)
        db = 16 if K else 0
        V = 10 * 4 ** case["level"] + 2
        fwd, bwd = 16 + db + 4 * a + 8 * K, 32 + 2 * db + 4 * a + 8 * K
        return {"bytes": (fwd + bwd) * P + 3.0 * case["n"] * V * a * 4,
                "flops": (20.0 * a + 20.0 * K) * P}
    if k == "tex":
        mip, c = "mipmap" in case["filter"], case["c"]
        t = case["th"] * case["tw"] * c * 4 * (4.0 / 3.0 if mip else 1.0)
        px = 8 + (16 if mip else 0) + (4 if case["bias"] == "map" else 0)
        return {"bytes": (3 * px + 8 * c) * P + 3 * t, "flops": (60.0 + 60.0 * c) * P}
    if k == "cube":
        return {"bytes": (24 + 8 * case["c"]) * P + 2.0 * 6 * case["size"] ** 2 * case["c"] * 4,
                "flops": (60.0 + 16.0 * case["c"]) * P}
    return {"bytes": (16 + 8 * case["c"] + 16 + 12 * case["c"]) * P + 2 * mesh,
            "flops": 100.0 * P}


# Largest relative error of a float32 result against the float64 one over the
# ranges above, times about four.  The gradients through triangle edges and
# depths (pos of fit, chain, peel, raster, aa) lose digits to cancellation in
# grazing triangles; texture coordinates of a tiled texture lose some to the
# repeat; sums alone stay near 1e-6.
_REL = {"fit": 4e-4, "chain": 1e-2, "peel": 1e-2, "range": 1e-3, "raster": 2e-2, "interp": 1e-5,
        "tex": 1e-3, "cube": 5e-5, "aa": 2e-2}


def tolerance(case):
    """`max` allows for single pixels on a switch (a mip level's end, an
    edge's sign), where the last bit decides between two values."""
    rel = _REL[case["kind"]]
    return {"rel": rel, "max": 0.5 if rel >= 1e-3 else 40 * rel}


# ---------------------------------------------------------------------------
# the same in float64
# ---------------------------------------------------------------------------

def cover(pos, tri, h, w):
    """Triangle shown at each pixel [N,h,w] (-1: none): the nearest of those
    whose edges include the centre, the lowest index at equal depth.  Decided
    in float32, each expression rounded as rasterize's definition states it:
    which of two triangles holds a centre on their edge is a choice, not a
    value, and everything behind it follows from that choice."""
    out = torch.full((pos.shape[0], h * w), -1, dtype=torch.int64, device=DEV)
    tri = tri.long()
    for n in range(pos.shape[0]):
        p = pos[n].float()[tri]  # [T,3,4]
        s = p[..., :3] / p[..., 3:]
        area = _cross(s[:, 1] - s[:, 0], s[:, 2] - s[:, 0])
        lo, hi = s[..., :2].amin(1), s[..., :2].amax(1)
        # a box a pixel wider than the triangle; the edge tests decide
        x0 = (torch.ceil((lo[:, 0] + 1) * w / 2 - 0.5) - 1).clamp(0, w).long()
        x1 = (torch.floor((hi[:, 0] + 1) * w / 2 - 0.5) + 1).clamp(-1, w - 1).long()
        y0 = (torch.ceil((1 - hi[:, 1]) * h / 2 - 0.5) - 1).clamp(0, h).long()
        y1 = (torch.floor((1 - lo[:, 1]) * h / 2 - 0.5) + 1).clamp(-1, h - 1).long()
        bw, bh = (x1 - x0 + 1).clamp_min(0), (y1 - y0 + 1).clamp_min(0)
        cnt = torch.where((area != 0) & (p[..., 3] > 0).all(1), bw * bh, torch.zeros_like(bw))
        t = torch.repeat_interleave(torch.arange(tri.shape[0], device=DEV), cnt)
        o = torch.arange(t.shape[0], device=DEV) - (cnt.cumsum(0) - cnt)[t]
        X, Y = x0[t] + o % bw[t], y0[t] + o // bw[t]
        # (full tensors: a division by a Python number becomes a product)
        px = 2.0 * (X.float() + 0.5) / torch.full_like(area, w)[t] - 1.0
        py = 1.0 - 2.0 * (Y.float() + 0.5) / torch.full_like(area, h)[t]
        d = s[t][..., :2] - torch.stack([px, py], -1)[:, None]
        e0, e1, e2 = _cross(d[:, 1], d[:, 2]), _cross(d[:, 2], d[:, 0]), _cross(d[:, 0], d[:, 1])
        ar, inv, sz = area[t], (1.0 / area)[t], s[t][..., 2]
        z = e0 * inv * sz[:, 0] + e1 * inv * sz[:, 1] + e2 * inv * sz[:, 2]
        ok = (e0 * ar >= 0) & (e1 * ar >= 0) & (e2 * ar >= 0) & (z >= -1) & (z <= 1) & \
            (px >= lo[t, 0]) & (px <= hi[t, 0]) & (py >= lo[t, 1]) & (py <= hi[t, 1])
        t, z, pix = t[ok], z[ok], (Y * w + X)[ok]
        best = torch.full((h * w,), 2.0, device=DEV).scatter_reduce_(0, pix, z, "amin")
        win = z == best[pix]
        first = torch.full((h * w,), 1 << 40, dtype=torch.int64, device=DEV)
        first.scatter_reduce_(0, pix[win], t[win], "amin")
        out[n] = torch.where(first < (1 << 40), first, out[n])
    return out.reshape(-1, h, w)


def _cross(a, b):
    return a[..., 0] * b[..., 1] - b[..., 0] * a[..., 1]


def _edges(s, px, py, area):
    """(e0, e1, e2) / area [M,3] and the depth at (px, py) of triangles s [M,3,3]."""
    x, y = s[..., 0] - px[:, None], s[..., 1] - py[:, None]
    e = torch.stack([x[:, 1] * y[:, 2] - x[:, 2] * y[:, 1], x[:, 2] * y[:, 0] - x[:, 0] * y[:, 2],
                     x[:, 0] * y[:, 1] - x[:, 1] * y[:, 0]], -1) / area[:, None]
    return e, (e * s[..., 2]).sum(-1)


def bary(pos, tri, tid, h, w):
    """rast and rast_db [N,h,w,4] of the shown triangles, differentiable in
    pos [N,V,4] (float64)."""
    n, Y, X = torch.nonzero(tid >= 0, as_tuple=True)
    t = tid[n, Y, X]
    p = pos[n[:, None], tri.long()[t]]
    s = p[..., :3] / p[..., 3:]
    x, y = s[..., 0], s[..., 1]
    area = (x[:, 1] - x[:, 0]) * (y[:, 2] - y[:, 0]) - (x[:, 2] - x[:, 0]) * (y[:, 1] - y[:, 0])
    e, z = _edges(s, 2 * (X + 0.5) / w - 1, 1 - 2 * (Y + 0.5) / h, area)
    kx, ky = 2.0 / w / area, -2.0 / h / area
    r = torch.stack([e[:, 1], e[:, 2], z, t + 1.0], -1)
    d = torch.stack([(y[:, 2] - y[:, 0]) * kx, (x[:, 0] - x[:, 2]) * ky,
                     (y[:, 0] - y[:, 1]) * kx, (x[:, 1] - x[:, 0]) * ky], -1)
    empty = torch.zeros(tid.shape + (4,), dtype=torch.float64, device=DEV)
    return empty.index_put((n, Y, X), r), empty.index_put((n, Y, X), d)


def interp64(attr, rast, db, tri, diff):
    """attr [1|N,V,A]; diff: attribute indices of the derivatives."""
    n, Y, X = torch.nonzero(rast[..., 3] > 0, as_tuple=True)
    r = rast[n, Y, X]
    v = tri.long()[r[:, 3].detach().round().long() - 1]
    a = attr[(n if attr.shape[0] > 1 else n * 0)[:, None], v]  # [M,3,A]
    u, w_ = r[:, 0:1], r[:, 1:2]
    o = (1 - u - w_) * a[:, 0] + u * a[:, 1] + w_ * a[:, 2]
    shape = tuple(rast.shape[:3])
    out = torch.zeros(shape + (attr.shape[-1],), dtype=torch.float64, device=DEV)
    out = out.index_put((n, Y, X), o)
    if not diff:
        return out, None
    d = db[n, Y, X]
    d1, d2 = (a[:, 1] - a[:, 0])[:, diff], (a[:, 2] - a[:, 0])[:, diff]
    da = torch.stack([d1 * d[:, 0:1] + d2 * d[:, 2:3], d1 * d[:, 1:2] + d2 * d[:, 3:4]], -1)
    oda = torch.zeros(shape + (2 * len(diff),), dtype=torch.float64, device=DEV)
    return out, oda.index_put((n, Y, X), da.reshape(da.shape[0], -1))


def _taps(tex, base, u, v, hk, wk, boundary):
    """Bilinear samples of flat texels tex [M,C] at u, v on levels of size
    (hk, wk) whose first texel is `base` (all per sample)."""
    x, y = u * wk - 0.5, v * hk - 0.5
    x0, y0 = torch.floor(x).detach(), torch.floor(y).detach()
    fx, fy = x - x0, y - y0
    out = 0
    for dy in (0, 1):
        for dx in (0, 1):
            xi, yi = x0.long() + dx, y0.long() + dy
            wgt = (fx if dx else 1 - fx) * (fy if dy else 1 - fy)
            if boundary == "zero":
                wgt = wgt * ((xi >= 0) & (xi < wk) & (yi >= 0) & (yi < hk))
            if boundary == "wrap":
                xi, yi = xi % wk, yi % hk
            else:
                xi, yi = torch.minimum(xi.clamp_min(0), wk - 1), torch.minimum(yi.clamp_min(0), hk - 1)
            out = out + wgt[:, None] * tex[base + yi * wk + xi]
    return out


def texture64(tex, uv, da, filt, boundary, bias=None, scalar=0.0):
    """tex [1,H,W,C]; uv [N,h,w,2]; da [N,h,w,4]."""
    shape, C = tuple(uv.shape[:3]), tex.shape[-1]
    u, v = uv.reshape(-1, 2).unbind(-1)
    H, W = tex.shape[1], tex.shape[2]
    full = lambda x: torch.full_like(u, x, dtype=torch.int64)  # noqa: E731
    if filt == "nearest":
        x, y = torch.floor(u * W).long(), torch.floor(v * H).long()
        inside = ((x >= 0) & (x < W) & (y >= 0) & (y < H)) if boundary == "zero" else \
            torch.ones_like(x, dtype=torch.bool)
        x, y = (x % W, y % H) if boundary == "wrap" else (x.clamp(0, W - 1), y.clamp(0, H - 1))
        return (tex.reshape(-1, C)[y * W + x] * inside[:, None]).reshape(shape + (C,))
    if filt == "linear":
        return _taps(tex.reshape(-1, C), full(0), u, v, full(H), full(W), boundary).reshape(
            shape + (C,))
    levels = [tex[0]]
    while levels[-1].shape[0] % 2 == 0 and levels[-1].shape[1] % 2 == 0:
        q = levels[-1]
        levels.append((q[0::2, 0::2] + q[0::2, 1::2] + q[1::2, 0::2] + q[1::2, 1::2]) / 4)
    L = len(levels)
    flat = torch.cat([q.reshape(-1, C) for q in levels])
    num = [q.shape[0] * q.shape[1] for q in levels]
    off = torch.tensor([sum(num[:i]) for i in range(L)], device=DEV)
    hs = torch.tensor([q.shape[0] for q in levels], device=DEV)
    ws = torch.tensor([q.shape[1] for q in levels], device=DEV)
    d = da.reshape(-1, 4) * 2.0 ** scalar
    if bias is not None:
        d = d * torch.exp2(bias.reshape(-1, 1))
    A = (d[:, 0] * W) ** 2 + (d[:, 2] * H) ** 2
    B = (d[:, 1] * W) ** 2 + (d[:, 3] * H) ** 2
    lod = (0.5 * torch.log2(torch.maximum(A, B).clamp_min(1e-20))).clamp(0, L - 1)
    tri_k0 = torch.floor(lod.detach()).long()
    tri_k1 = (tri_k0 + 1).clamp_max(L - 1)
    if filt == "linear-mipmap-linear":
        s0 = _taps(flat, off[tri_k0], u, v, hs[tri_k0], ws[tri_k0], boundary)
        s1 = _taps(flat, off[tri_k1], u, v, hs[tri_k1], ws[tri_k1], boundary)
        f = (lod - tri_k0)[:, None]
        return ((1 - f) * s0 + f * s1).reshape(shape + (C,))
    k = torch.floor(lod.detach() + 0.5).long().clamp_max(L - 1)
    out = _taps(flat, off[k], u, v, hs[k], ws[k], boundary)
    # mip-nearest: the derivatives take the trilinear blend's LOD gradient
    with torch.no_grad():
        s0 = _taps(flat, off[tri_k0], u, v, hs[tri_k0], ws[tri_k0], boundary)
        s1 = _taps(flat, off[tri_k1], u, v, hs[tri_k1], ws[tri_k1], boundary)
    f = (lod - lod.detach())[:, None]
    return (out + f * (s1 - s0)).reshape(shape + (C,))


def cube64(tex, dirs):
    """Bilinear lookup of tex [1,6,S,S,C] along dirs [N,h,w,3]."""
    shape, S, C = tuple(dirs.shape[:3]), tex.shape[2], tex.shape[-1]
    x, y, z = dirs.reshape(-1, 3).unbind(-1)
    ax, ay, az = x.abs(), y.abs(), z.abs()
    mx, my = (ax >= ay) & (ax >= az), ay >= az
    pick = lambda a, b, c: torch.where(mx, a, torch.where(my, b, c))  # noqa: E731
    one = torch.ones_like(x)
    face = pick(torch.where(x > 0, 0, 1), torch.where(y > 0, 2, 3), torch.where(z > 0, 4, 5))
    sc = pick(torch.where(x > 0, -z, z), x, torch.where(z > 0, x, -x))
    tc = pick(-y, torch.where(y > 0, z, -z), -y)
    ma = pick(ax, ay, az)
    size = (one * S).long()
    return _taps(tex.reshape(-1, C), face * S * S, (sc / ma + 1) / 2, (tc / ma + 1) / 2, size, size,
                 "clamp").reshape(shape + (C,))


def topology64(tri):
    """Triangle across the edge opposite each vertex (-1 boundary, -2 shared
    by three or more)."""
    T = tri.shape[0]
    a, b = tri.long()[:, [1, 2, 0]].reshape(-1), tri.long()[:, [2, 0, 1]].reshape(-1)
    _, inv, cnt = torch.unique(torch.minimum(a, b) * (1 << 32) + torch.maximum(a, b),
                               return_inverse=True, return_counts=True)
    total = torch.zeros_like(cnt).scatter_add_(0, inv, torch.arange(3 * T, device=DEV) // 3)
    other = total[inv] - torch.arange(3 * T, device=DEV) // 3
    c = cnt[inv]
    return torch.where(c == 2, other, torch.where(c == 1, -1, -2)).reshape(T, 3)


def aa64(color, tid, pos, tri):
    """color [N,h,w,C] blended across the edges that separate neighbouring
    pixels' triangles; pos [N,V,4]."""
    N, h, w, _ = color.shape
    topo, tri = topology64(tri), tri.long()
    out = color
    for dy, dx in ((0, 1), (1, 0), (0, -1), (-1, 0)):
        nb = torch.full_like(tid, -9)
        ys, xs = slice(max(0, -dy), h - max(0, dy)), slice(max(0, -dx), w - max(0, dx))
        yn, xn = slice(max(0, dy), h - max(0, -dy)), slice(max(0, dx), w - max(0, -dx))
        nb[:, ys, xs] = tid[:, yn, xn]
        n, Y, X = torch.nonzero((nb != -9) & (nb != tid), as_tuple=True)
        tp, tn = tid[n, Y, X], nb[n, Y, X]
        fg = torch.where(tp >= 0, tp, tn)
        target = torch.where(tp >= 0, tn, -1)
        p = pos[n[:, None], tri[fg]]
        ex = (p[..., 0] / p[..., 3] + 1) * w / 2
        ey = (1 - p[..., 1] / p[..., 3]) * h / 2
        px, py = X + 0.5, Y + 0.5
        found = torch.zeros_like(n, dtype=torch.bool)
        edge = torch.zeros_like(n)
        for kk in range(3):
            x0, y0 = ex[:, (kk + 1) % 3], ey[:, (kk + 1) % 3]
            vx, vy = ex[:, (kk + 2) % 3] - x0, ey[:, (kk + 2) % 3] - y0
            sp = vx * (py - y0) - vy * (px - x0)
            sn = vx * (py + dy - y0) - vy * (px + dx - x0)
            hit = ~found & (topo[fg, kk] == target) & (sp * sn < 0)
            edge = torch.where(hit, kk, edge)
            found = found | hit
        n, Y, X, ex, ey, edge = (q[found] for q in (n, Y, X, ex, ey, edge))
        i = torch.arange(n.shape[0], device=DEV)
        x0, y0 = ex[i, (edge + 1) % 3], ey[i, (edge + 1) % 3]
        x1, y1 = ex[i, (edge + 2) % 3], ey[i, (edge + 2) % 3]
        if dy == 0:
            (p0, p1, q0, q1), at, c, first = (x0, x1, y0, y1), Y + 0.5, X + 0.5, X
        else:
            (p0, p1, q0, q1), at, c, first = (y0, y1, x0, x1), X + 0.5, Y + 0.5, Y
        den = q1 - q0
        safe = den.abs() >= 1e-7
        t = (at - q0) / torch.where(safe, den, torch.ones_like(den))
        cross = p0 + t * (p1 - p0)
        on = safe & (t >= 0) & (t <= 1) & (cross > first) & (cross < first + 1)
        alpha = torch.where(on, (0.5 - (cross - c).abs()).clamp_min(0), torch.zeros_like(cross))
        diff = color[n, Y + dy, X + dx] - color[n, Y, X]
        out = out + torch.zeros_like(color).index_put((n, Y, X), alpha[:, None] * diff)
    return out


def exact(case, seed):
    k, h, w = case["kind"], case["h"], case["w"]
    if k in ("peel", "range"):
        return None  # minutes of float64 work at these sizes
    s = _inputs(case, seed)
    s = {name: v.double() if v.is_floating_point() else v for name, v in s.items()}
    leaves = [name for name in _leaves(case) if name in s]
    for name in leaves:
        s[name].requires_grad_(True)
    grads = None
    if k in ("fit", "chain"):
        tid = cover(s["pos"].detach(), s["tri"], h, w)
        rast, db = bary(s["pos"], s["tri"], tid, h, w)
        attr = s["attr"] if s["attr"].ndim == 3 else s["attr"][None]
        if k == "fit":
            out, _ = interp64(attr, rast, None, s["tri"], [])
        else:
            uv, da = interp64(attr, rast, db, s["tri"], [0, 1])
            out = texture64(s["tex"], uv, da, "linear-mipmap-linear", "clamp")
        if k == "chain" or case["mesh"] == "pie":
            out = aa64(out, tid, s["pos"], s["tri"])
        outs = {"loss": ((out - s["target"]) ** 2).mean(), "image": out}
    elif k == "raster":
        rast, db = bary(s["pos"], s["tri"], cover(s["pos"].detach(), s["tri"], h, w), h, w)
        outs, grads = {"rast": rast, "rast_db": db}, [s["g"], s["gdb"]]
    elif k == "interp":
        diff = list(range(case["a"])) if case["diff"] == "all" else \
            [int(i) for i in case["diff"].split(",")] if case["diff"] else []
        out, da = interp64(s["attr"], s["rast"], s["rast_db"], s["tri"], diff)
        outs, grads = ({"out": out, "out_da": da}, [s["g"], s["gda"]]) if diff else \
            ({"out": out}, [s["g"]])
    elif k == "tex":
        outs = {"out": texture64(s["tex"], s["uv"], s.get("uv_da"), case["filter"],
                                 case["boundary"], s.get("bias"),
                                 0.5 if case["bias"] == "scalar" else 0.0)}
        grads = [s["g"]]
    elif k == "cube":
        outs, grads = {"out": cube64(s["tex"], s["uv"])}, [s["g"]]
    else:
        tid = s["rast"][..., 3].round().long() - 1
        outs, grads = {"out": aa64(s["color"], tid, s["pos"], s["tri"])}, [s["g"]]
    heads = [outs["loss"]] if "loss" in outs else list(outs.values())
    got = torch.autograd.grad(heads, [s[name] for name in leaves], grads, allow_unused=True)
    outs.update(("d_" + name, v if v is not None else torch.zeros_like(s[name]))
                for name, v in zip(leaves, got))
    return {name: v.detach() for name, v in outs.items()}
