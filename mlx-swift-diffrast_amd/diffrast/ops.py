"""`DiffRast`: the four differentiable rasterization ops on MI355X.

Mirrors the public API of mnmly/mlx-swift-diffrast (the `DiffRast` enum in
Sources/MLXDiffRast/*.swift): same op names, argument names and meanings,
output layouts and conventions (clip-space pos, rast = (u, v, z/w,
tri_id+1), rastDB, instanced / range modes, top-left pixel origin).  Each op
is a compiled autograd node (csrc/torch_ops.cpp) whose forward and backward
call the C ABI of libdiffrast_mi355x.so, the counterpart of the reference's
`CustomFunction { Forward; VJP }` pairs; this module turns arguments into
tensors and names into modes.  Swift `precondition` failures become
`ValueError`.

Tensors live on the current ROCm device; there is no CPU path.
"""
from __future__ import annotations

import ctypes
import enum
from typing import List, Optional, Sequence, Tuple, Union

import torch

from . import _lib


class BoundaryMode(enum.IntEnum):
    """Texture.swift:8-17."""
    wrap = 0
    clamp = 1
    zero = 2
    cube = 3


class FilterMode(enum.IntEnum):
    """Texture.swift:35-40."""
    nearest = 0
    linear = 1
    linearMipmapNearest = 2
    linearMipmapLinear = 3


_FILTER_NAMES = {"nearest": 0, "linear": 1, "linear-mipmap-nearest": 2,
                 "linear-mipmap-linear": 3, "linearMipmapNearest": 2, "linearMipmapLinear": 3}
_BOUNDARY_NAMES = {"wrap": 0, "clamp": 1, "zero": 2, "cube": 3}


class DiffAttrs:
    """Interpolate.swift:15-18: `DiffAttrs.all` or `DiffAttrs.indices([...])`."""

    def __init__(self, indices: Optional[Sequence[int]] = None):
        self.idx = None if indices is None else [int(i) for i in indices]

    @classmethod
    def indices(cls, idx: Sequence[int]) -> "DiffAttrs":
        return cls(list(idx))

    def __eq__(self, other):
        return isinstance(other, DiffAttrs) and self.idx == other.idx

    def __repr__(self):
        return "DiffAttrs.all" if self.idx is None else f"DiffAttrs.indices({self.idx})"


DiffAttrs.all = DiffAttrs(None)


def _ptr(t: Optional[torch.Tensor]):
    return None if t is None else ctypes.c_void_p(t.data_ptr())


# The current stream's handle.  torch.cuda.current_stream() builds a Stream
# object per call (~10 us, several calls per op); the raw query returns the
# same handle directly.
if hasattr(torch._C, "_cuda_getCurrentRawStream") and hasattr(torch._C, "_cuda_getDevice"):
    _raw_stream = torch._C._cuda_getCurrentRawStream
    _cur_device = torch._C._cuda_getDevice
else:
    def _raw_stream(index):
        return torch.cuda.current_stream(index).cuda_stream
    _cur_device = torch.cuda.current_device


def _stream():
    return ctypes.c_void_p(_raw_stream(_cur_device()))


def _tensor(t) -> torch.Tensor:
    return t if isinstance(t, torch.Tensor) else torch.as_tensor(t)


def _dev_f32(t: torch.Tensor, name: str) -> torch.Tensor:
    if not isinstance(t, torch.Tensor) or not t.is_cuda:
        raise ValueError(f"{name} must be a tensor on a ROCm device")
    return t.detach().to(torch.float32).contiguous()


def _dev_i32(t, name: str, device) -> torch.Tensor:
    if not isinstance(t, torch.Tensor):
        t = torch.as_tensor(t)
    return t.detach().to(device=device, dtype=torch.int32).contiguous()


class MipPyramid(list):
    """What `textureConstructMip` returns: the list [tex, level1, ...] plus
    the identity and in-place version of `tex` when the levels were built,
    so that `texture(mip=...)` can refuse a pyramid whose texture has been
    changed since (an optimizer step updates it in place)."""

    def __init__(self, levels, tex):
        super().__init__(levels)
        self.source_ptr = tex.data_ptr()
        self.source_version = tex._version


def _packed_pyramid(levels, tex):
    """(L, packed levels 1..L-1) of a `textureConstructMip` list: its levels
    are views of one buffer in the library's packing, used as they are; any
    other list of [Nt, Hk, Wk, C] levels is packed by a copy.  A
    `MipPyramid` must still describe `tex` as it is now."""
    if isinstance(levels, MipPyramid):
        if tex.data_ptr() != levels.source_ptr:
            raise ValueError("texture: mip was built from another texture tensor "
                             "(textureConstructMip(tex) of the tex passed here)")
        if tex._version != levels.source_version:
            raise ValueError("texture: tex was modified in place after textureConstructMip; "
                             "rebuild mip from the current texture")
    levels = list(levels)
    if not levels:
        raise ValueError("texture: mip must hold at least level 0")
    Nt, H, W, C = tex.shape
    if tuple(levels[0].shape) != (Nt, H, W, C):
        raise ValueError(f"texture: mip[0] must be the texture's shape {[Nt, H, W, C]}")
    h, w = H, W
    for k, lv in enumerate(levels[1:], 1):
        h, w = h // 2, w // 2
        if tuple(lv.shape) != (Nt, h, w, C) or not lv.is_cuda:
            raise ValueError(f"texture: mip[{k}] must be [{Nt}, {h}, {w}, {C}] on the device "
                             f"(got {list(lv.shape)})")
    L = len(levels)
    if L > 1 and h < 1:
        raise ValueError("texture: mip has more levels than the texture allows")
    if L == 1:
        return 1, torch.empty(1, device=tex.device, dtype=torch.float32)
    first = levels[1]
    packed = all(lv.dtype == torch.float32 and lv.is_contiguous() for lv in levels[1:])
    off = 0
    for lv in levels[1:]:
        if not packed or lv.data_ptr() != first.data_ptr() + 4 * off:
            packed = False
            break
        off += lv.numel()
    if packed:
        n = sum(lv.numel() for lv in levels[1:])
        return L, first.reshape(-1).as_strided((n,), (1,))
    return L, torch.cat([lv.detach().to(torch.float32).reshape(-1) for lv in levels[1:]])


# ---------------------------------------------------------------------------
# public API
# ---------------------------------------------------------------------------

class DiffRast:
    """Namespace of the ops (MLXDiffRast.swift:18)."""

    BoundaryMode = BoundaryMode
    FilterMode = FilterMode
    DiffAttrs = DiffAttrs

    @staticmethod
    def rasterize(pos: torch.Tensor, tri, resolution: Tuple[int, int], gradDB: bool = True,
                  ranges=None, peelLayer: Optional[torch.Tensor] = None, maxPerTile: int = 0
                  ) -> Tuple[torch.Tensor, torch.Tensor]:
        """Rasterize.swift:44-144.  Instanced pos [N,V,4], or range mode: pos
        [V,4] with ranges [N,2] (start, count) per image.  Returns (rast,
        rastDB); rastDB is [N,H,W,0] when gradDB is False.

        `ranges` is read on the host (a device tensor is copied back first,
        which waits for it).  `maxPerTile` (no counterpart argument in the
        reference): 0 keeps every triangle; 128 reproduces the reference's
        per-tile limit (MAX_PER_TILE, Rasterize.swift:164-171), each 16x16
        tile keeping its 128 lowest triangle indices (the reference keeps
        the first 128 of its atomic appends)."""
        H, W = int(resolution[0]), int(resolution[1])
        if not isinstance(pos, torch.Tensor):
            raise ValueError("rasterize: pos must be a tensor on a ROCm device")
        if peelLayer is not None and not isinstance(peelLayer, torch.Tensor):
            raise ValueError("peelLayer must be a tensor on a ROCm device")
        if ranges is not None:
            ranges = (ranges.detach().cpu() if isinstance(ranges, torch.Tensor)
                      else torch.as_tensor(ranges)).to(torch.int32).contiguous()
        return _lib.ops().rasterize(pos, _tensor(tri), H, W, bool(gradDB), ranges, peelLayer,
                                    int(maxPerTile))

    @staticmethod
    def rasterizeTileCounts(pos: torch.Tensor, tri, resolution: Tuple[int, int],
                            ranges=None) -> torch.Tensor:
        """Binning report: per 16x16 tile, the number of triangles binned to
        it, [N, ceil(H/16), ceil(W/16)] int32 -- the reference's bin counts
        (Rasterize.swift:227-239).  Tiles above 128 are those where the
        reference drops triangles (MAX_PER_TILE, :164-171); rasterize here
        keeps them all.  Same layouts as `rasterize`."""
        H, W = int(resolution[0]), int(resolution[1])
        posf = _dev_f32(pos.detach() if isinstance(pos, torch.Tensor) else pos,
                        "rasterizeTileCounts: pos")
        tri32 = _dev_i32(tri, "tri", posf.device)
        if tri32.ndim != 2 or tri32.shape[1] != 3:
            raise ValueError(f"rasterizeTileCounts: tri must be [T, 3] (got {list(tri32.shape)})")
        rng = None
        if ranges is not None:
            if posf.ndim != 2 or posf.shape[1] != 4:
                raise ValueError("rasterizeTileCounts: with `ranges`, pos must be [V, 4]")
            r = ranges.detach().cpu() if isinstance(ranges, torch.Tensor) else torch.as_tensor(ranges)
            rng = r.to(torch.int32).contiguous().numpy()
            if rng.ndim != 2 or rng.shape[1] != 2:
                raise ValueError("rasterizeTileCounts: ranges must be [N, 2]")
            N, V = rng.shape[0], posf.shape[0]
        else:
            if posf.ndim != 3 or posf.shape[2] != 4:
                raise ValueError("rasterizeTileCounts: pos must be [N, V, 4]")
            N, V = posf.shape[0], posf.shape[1]
        lib = _lib.load()
        counts = torch.empty((N, (H + 15) // 16, (W + 15) // 16), device=posf.device,
                             dtype=torch.int32)
        _lib.check(lib.dr_rasterize_tile_counts(
            _ptr(posf), 0 if rng is not None else V * 4, _ptr(tri32),
            rng.ctypes.data_as(ctypes.c_void_p) if rng is not None else None, N, V,
            tri32.shape[0], H, W, _ptr(counts), None, _stream()))
        return counts

    @staticmethod
    def interpolate(attr: torch.Tensor, rast: torch.Tensor, tri, rastDB=None,
                    diffAttrs: Union[None, DiffAttrs, str, Sequence[int]] = None
                    ) -> Tuple[torch.Tensor, torch.Tensor]:
        """Interpolate.swift:43-132.  attr [V,A], [1,V,A] or [N,V,A]."""
        if isinstance(diffAttrs, str):
            if diffAttrs != "all":
                raise ValueError("interpolate: diffAttrs must be 'all' or indices")
            mode, idx = 1, []
        elif diffAttrs is None:
            mode, idx = 0, []
        else:
            idx = diffAttrs.idx if isinstance(diffAttrs, DiffAttrs) else [int(i) for i in diffAttrs]
            mode, idx = (1, []) if idx is None else (2, idx)
        return _lib.ops().interpolate(attr, rast, _tensor(tri), rastDB, mode, idx)

    @staticmethod
    def texture(tex: torch.Tensor, uv: torch.Tensor, uvDA: Optional[torch.Tensor] = None,
                filterMode: Union[FilterMode, str] = FilterMode.linear,
                boundaryMode: Union[BoundaryMode, str] = BoundaryMode.wrap,
                mipLevelBias: float = 0.0, mipLevelBiasMap: Optional[torch.Tensor] = None,
                mip: Optional[Sequence[torch.Tensor]] = None, dirGrad: bool = False
                ) -> torch.Tensor:
        """Texture.swift:62-131.

        `mip` (mip filters only; no counterpart argument in the reference):
        a pyramid `[tex, level1, ...]` from `textureConstructMip(tex)`, kept
        across calls with the same texture so it is not rebuilt
        (Texture.swift:141-143 suggests such caching).  Its levels are read
        as given (fewer levels cap the LOD); the gradient still flows to
        `tex` through the 2x2 box backward, as for a pyramid built in the
        call.  A pyramid from `textureConstructMip` raises ValueError once
        `tex` has been changed in place (or when another tensor is passed);
        a plain list of levels is taken as it is.

        Cube maps (boundaryMode cube) also take the mip filters, with uvDA
        the direction's screen derivatives [N, H_img, W_img, 6] (the layout
        `interpolate(..., diffAttrs=.all)` gives a 3-channel direction), and
        `dirGrad=True` returns the direction gradient instead of the
        reference's zeros (Texture.swift:196-198).  Both are extensions; the
        reference samples cube maps bilinearly only (:75-76)."""
        filt = FilterMode(_FILTER_NAMES[filterMode] if isinstance(filterMode, str) else filterMode)
        bnd = BoundaryMode(_BOUNDARY_NAMES[boundaryMode] if isinstance(boundaryMode, str)
                           else boundaryMode)
        levels, pyramid = 0, None
        if mip is not None and (bnd == BoundaryMode.cube or filt >= FilterMode.linearMipmapNearest):
            if bnd == BoundaryMode.cube:
                raise ValueError("texture: a prebuilt `mip` is for 2D textures")
            levels, pyramid = _packed_pyramid(mip, tex)
        return _lib.ops().texture(tex, uv, uvDA, int(filt), int(bnd), float(mipLevelBias),
                                  mipLevelBiasMap, levels, pyramid, bool(dirGrad))

    @staticmethod
    def textureConstructMip(tex: torch.Tensor, maxLevel: Optional[int] = None) -> List[torch.Tensor]:
        """Texture.swift:144-161: [level0 = tex, level1, ...], 2x2 box means
        (a `MipPyramid`, which also records tex's in-place version)."""
        if tex.ndim != 4:
            raise ValueError(f"textureConstructMip: tex must be [N, H, W, C] (got {list(tex.shape)})")
        lib = _lib.load()
        Nt, H, W, C = tex.shape
        L = lib.dr_texture_mip_levels(H, W, -1 if maxLevel is None else int(maxLevel), None, None)
        texf = _dev_f32(tex, "textureConstructMip: tex")
        size = lib.dr_texture_mip_size(Nt, H, W, C, L)
        pyr = torch.empty(max(size, 1), device=texf.device, dtype=torch.float32)
        _lib.check(lib.dr_texture_build_mip(_ptr(texf), Nt, H, W, C, L, _ptr(pyr), _stream()))
        levels, off, h, w = [tex], 0, H, W
        for _ in range(1, L):
            h, w = h // 2, w // 2
            n = Nt * h * w * C
            levels.append(pyr[off:off + n].view(Nt, h, w, C))
            off += n
        return MipPyramid(levels, tex)

    @staticmethod
    def antialiasConstructTopologyHash(tri) -> torch.Tensor:
        """Antialias.swift:19-66, computed on the GPU."""
        tri32 = _dev_i32(tri, "tri", torch.device("cuda", torch.cuda.current_device())
                         if not isinstance(tri, torch.Tensor) or not tri.is_cuda else tri.device)
        if tri32.ndim != 2 or tri32.shape[1] != 3:
            raise ValueError("antialiasConstructTopologyHash: tri must be [T, 3] "
                             f"(got {list(tri32.shape)})")
        lib = _lib.load()
        topo = torch.empty_like(tri32)
        _lib.check(lib.dr_antialias_topology(_ptr(tri32), tri32.shape[0], _ptr(topo), _stream()))
        return topo

    @staticmethod
    def antialias(color: torch.Tensor, rast: torch.Tensor, pos: torch.Tensor, tri,
                  topologyHash: Optional[torch.Tensor] = None) -> torch.Tensor:
        """Antialias.swift:90-131."""
        return _lib.ops().antialias(color, rast, pos, _tensor(tri),
                                    None if topologyHash is None else _tensor(topologyHash))


rasterize = DiffRast.rasterize
interpolate = DiffRast.interpolate
texture = DiffRast.texture
textureConstructMip = DiffRast.textureConstructMip
antialiasConstructTopologyHash = DiffRast.antialiasConstructTopologyHash
antialias = DiffRast.antialias
