"""texture's backward paths on smooth uv fields (what a rendered surface
gives), against the CPU oracle, at the sizes where a path changes: wrap
windows across the texture's border and repeats; boxes that fill the LDS
pool, take it in bands, or are written to memory directly; more than four
channels (chunks of four, remainders, one pool pass or several, the channel
limit); pyramids of sizes that are no multiple of a patch."""
import numpy as np
import pytest

import oracle as O
from parity import assert_fwd_close, assert_grad_close, dev, host, torch_dev

pytestmark = pytest.mark.gpu


def smooth_uv(rng, N, Hi, Wi, scale, offset, background):
    """An affine field over `scale` repeats from `offset`, its derivatives,
    and a patch and single pixels of one constant uv (empty pixels)."""
    y, x = np.meshgrid((np.arange(Hi) + 0.5) / Hi, (np.arange(Wi) + 0.5) / Wi, indexing="ij")
    M = rng.normal(size=(N, 2, 2)) * scale
    uv = np.stack([np.stack([M[n, 0, 0] * x + M[n, 0, 1] * y, M[n, 1, 0] * x + M[n, 1, 1] * y], -1)
                   for n in range(N)]) + offset
    da = np.stack([np.broadcast_to([M[n, 0, 0] / Wi, M[n, 0, 1] / Hi, M[n, 1, 0] / Wi,
                                    M[n, 1, 1] / Hi], (Hi, Wi, 4)) for n in range(N)]).copy()
    empty = np.zeros((N, Hi, Wi), bool)
    empty[:, : Hi // 2, : Wi // 3] = True
    empty[:, ::7, ::5] = True
    uv[empty], da[empty] = background, 0.0
    return uv.astype(np.float32), da.astype(np.float32)


def check(rng, tex, uv, da, filt, bnd, rtol=1e-4, bias=None):
    from diffrast import DiffRast
    mip = "mipmap" in filt
    t, u = dev(tex).requires_grad_(True), dev(uv).requires_grad_(True)
    d = dev(da).requires_grad_(True) if mip else None
    kw = dict(filterMode=filt, boundaryMode=bnd)
    if bias is not None:
        kw["mipLevelBias"] = bias
    out = DiffRast.texture(t, u, uvDA=d, **kw)
    ref = O.texture(tex, uv, uvDA=da if mip else None, **kw)
    assert_fwd_close(host(out), ref)
    g = rng.normal(size=ref.shape).astype(np.float32)
    out.backward(dev(g))
    d_tex, d_uv, d_da, _ = O.texture_vjp(tex, uv, g, uvDA=da if mip else None, **kw)
    assert_grad_close(host(t.grad), d_tex, "d_tex", rtol=rtol)
    assert_grad_close(host(u.grad), d_uv, "d_uv", rtol=rtol)
    if mip:
        assert_grad_close(host(d.grad), d_da, "d_uvDA", rtol=rtol)


# texture sizes of one texel a side, odd ones, one smaller and one larger
# than a tile's footprint; offsets beyond the packed window coordinates
# (taken wrapped) and around zero; the background at uv (0, 0) (four corner
# texels in wrap mode) and at another constant
@pytest.mark.parametrize("Ht,Wt", [(1, 1), (1, 7), (5, 3), (40, 72), (512, 256)])
@pytest.mark.parametrize("offset,background", [(0.0, (0.0, 0.0)), (-3.5, (0.3, 0.7)),
                                               (40000.0, (0.0, 0.0))])
@pytest.mark.parametrize("filt,C", [("linear", 1), ("linear", 3), ("linear-mipmap-linear", 4),
                                    ("nearest", 2)])
def test_wrap_windows(Ht, Wt, offset, background, filt, C):
    torch_dev()
    rng = np.random.default_rng(Ht * 1000 + Wt + C)
    uv, da = smooth_uv(rng, 2, 35, 53, 1.5, offset, background)
    tex = rng.random((1, Ht, Wt, C)).astype(np.float32)
    check(rng, tex, uv, da, filt, "wrap")


# texels a pixel: a tile's box of 16 x 16 pixels grows from one window (0.5)
# over several bands (2 to 4) to the direct way (12); C = 4 has a smaller pool
@pytest.mark.parametrize("texels", [0.5, 2.0, 3.0, 4.0, 12.0])
@pytest.mark.parametrize("bnd", ["wrap", "clamp", "zero"])
@pytest.mark.parametrize("filt,C", [("linear", 1), ("linear", 3), ("linear", 4), ("nearest", 3),
                                    ("linear-mipmap-linear", 2)])
def test_minified_boxes(texels, bnd, filt, C):
    torch_dev()
    rng = np.random.default_rng(int(texels * 10) + C)
    Hi, Wi, Ht, Wt = 49, 60, 256, 320
    scale = texels * Wi / Wt / 1.5
    uv, da = smooth_uv(rng, 2, Hi, Wi, scale, 0.4, (0.0, 0.0))
    if "mipmap" in filt:  # the LOD of a magnified surface: level 0 at any footprint spread
        da *= 1e-3
    tex = rng.random((1, Ht, Wt, C)).astype(np.float32)
    check(rng, tex, uv, da, filt, bnd)


# channels: the first past the four-channel kernels, whole chunks, a pool
# filled exactly and in several passes, the limit of the empty pixels' sums
# and one beyond (the general kernel)
@pytest.mark.parametrize("C", [5, 8, 16, 23, 128, 129])
@pytest.mark.parametrize("filt,bnd", [("nearest", "wrap"), ("linear", "wrap"), ("linear", "zero"),
                                      ("linear-mipmap-linear", "clamp"),
                                      ("linear-mipmap-nearest", "wrap")])
@pytest.mark.parametrize("Nt,texels", [(1, 0.7), (2, 6.0)])
def test_many_channels(C, filt, bnd, Nt, texels):
    torch_dev()
    rng = np.random.default_rng(C * 10 + Nt)
    Hi, Wi, Ht, Wt = 35, 38, 64, 96
    uv, da = smooth_uv(rng, 2, Hi, Wi, texels * Wi / Wt / 1.5, 0.3, (0.0, 0.0))
    if "mipmap" in filt:
        da *= 0.6  # off whole LODs (a switch)
    tex = rng.random((Nt, Ht, Wt, C)).astype(np.float32)
    check(rng, tex, uv, da, filt, bnd, bias=0.3 if "mipmap" in filt else None)


@pytest.mark.parametrize("C", [1, 3, 4, 6, 9])
def test_smooth_cube(C):
    torch_dev()
    from diffrast import DiffRast
    rng = np.random.default_rng(C)
    tex = rng.random((1, 6, 24, 24, C)).astype(np.float32)
    y, x = np.meshgrid(np.linspace(-2, 2, 33), np.linspace(-2, 2, 40), indexing="ij")
    dirs = np.stack([np.stack([x, y, np.full_like(x, z)], -1) for z in (0.7, -1.1)])
    dirs = dirs.astype(np.float32)  # smooth, across the faces' edges
    t, u = dev(tex).requires_grad_(True), dev(dirs).requires_grad_(True)
    out = DiffRast.texture(t, u, boundaryMode="cube")
    np.testing.assert_array_equal(host(out), O.texture(tex, dirs, boundaryMode="cube"))
    g = rng.normal(size=out.shape).astype(np.float32)
    out.backward(dev(g))
    assert_grad_close(host(t.grad), O.texture_vjp(tex, dirs, g, boundaryMode="cube")[0], "d_tex")
    assert not host(u.grad).any()


@pytest.mark.parametrize("H,W", [(2, 2), (34, 66), (100, 40), (96, 32)])
@pytest.mark.parametrize("C", [3, 4, 6])
def test_pyramid_sizes(H, W, C):
    torch_dev()
    from diffrast import DiffRast
    tex = np.random.default_rng(C).random((2, H, W, C)).astype(np.float32)
    got, ref = DiffRast.textureConstructMip(dev(tex)), O.textureConstructMip(tex)
    assert len(got) == len(ref)
    for a, b in zip(got, ref):
        np.testing.assert_array_equal(host(a), b)


# scattered uv over a tiled texture: a tile's box is up to 49,152 texels on a
# side, more than 2^31 of them together
@pytest.mark.parametrize("filt,C", [("linear", 1), ("linear", 3), ("linear", 4), ("linear", 6),
                                    ("nearest", 1), ("nearest", 3), ("nearest", 6),
                                    ("linear-mipmap-linear", 3), ("linear-mipmap-linear", 4),
                                    ("linear-mipmap-nearest", 4), ("linear-mipmap-linear", 6)])
def test_scattered_wrap(filt, C):
    torch_dev()
    rng = np.random.default_rng(C)
    S = 2048
    uv = rng.uniform(-12.0, 12.0, size=(2, 17, 33, 2)).astype(np.float32)
    uv[:, :8] *= np.float32(0.01)  # and a part whose boxes fit
    da = rng.uniform(0.9, 1.1, size=(2, 17, 33, 4)).astype(np.float32) * np.float32(1.1 / S)
    tex = rng.random((1, S, S, C)).astype(np.float32)
    check(rng, tex, uv, da, filt, "wrap")


def nonfinite(rng, g):
    """g with a few infinities and NaNs."""
    g = g.copy()
    flat = g.reshape(-1)
    at = rng.choice(flat.size, size=24, replace=False)
    flat[at[:9]], flat[at[9:18]], flat[at[18:]] = np.inf, -np.inf, np.nan
    return g


def assert_same_nonfinite(got, ref, what):
    """NaN and infinities where the oracle has them, close elsewhere."""
    np.testing.assert_array_equal(np.isnan(got), np.isnan(ref), err_msg=what)
    np.testing.assert_array_equal(got[np.isinf(ref)], ref[np.isinf(ref)], err_msg=what)
    fin = np.isfinite(ref)
    assert_grad_close(got[fin], ref[fin], what)


# a cotangent that is not finite reaches the texel that was sampled and no
# other; outside the zero boundary's image it is masked to 0 * inf
@pytest.mark.parametrize("C", [1, 3, 4, 6, 129])
@pytest.mark.parametrize("bnd", ["wrap", "clamp", "zero"])
@pytest.mark.parametrize("texels", [0.3, 3.0, 12.0])
def test_nearest_nonfinite_cotangent(C, bnd, texels):
    torch_dev()
    from diffrast import DiffRast
    rng = np.random.default_rng(C)
    Hi, Wi, Ht, Wt = 33, 50, 160, 192
    uv, _ = smooth_uv(rng, 2, Hi, Wi, texels * Wi / Wt / 1.5, 0.2, (0.0, 0.0))
    tex = rng.random((1, Ht, Wt, C)).astype(np.float32)
    g = nonfinite(rng, rng.normal(size=(2, Hi, Wi, C)).astype(np.float32))
    t = dev(tex).requires_grad_(True)
    DiffRast.texture(t, dev(uv), filterMode="nearest", boundaryMode=bnd).backward(dev(g))
    ref = O.texture_vjp(tex, uv, g, filterMode="nearest", boundaryMode=bnd)[0]
    assert_same_nonfinite(host(t.grad), ref, "d_tex")


# cotangents that are not finite on footprints at texel centres, whose taps
# of weight zero (0 * inf) lie outside the boxes of the weighted ones
@pytest.mark.parametrize("C,bnd,filt", [(1, "wrap", "linear"), (3, "wrap", "linear"),
                                        (4, "wrap", "linear-mipmap-linear"), (3, "cube", "linear"),
                                        (6, "wrap", "linear"), (6, "clamp", "linear"),
                                        (6, "zero", "linear"), (6, "cube", "linear"),
                                        (6, "clamp", "linear-mipmap-linear")])
@pytest.mark.parametrize("step", [1, 4, 16])  # texels a pixel
@pytest.mark.parametrize("uv_grad", [False, True])
def test_zero_weight_taps_nonfinite_cotangent(C, bnd, filt, step, uv_grad):
    torch_dev()
    from diffrast import DiffRast
    rng = np.random.default_rng(C + step)
    Hi = Wi = 33
    S = 256
    i = (np.arange(Hi) * step + 40) % S  # (no texel at a border, where taps merge)
    y, x = np.meshgrid(i, i, indexing="ij")
    if bnd == "cube":  # exact in fp32: every quotient is by 1
        y, x = np.clip(y, 1, S - 2), np.clip(x, 1, S - 2)
        uv = np.stack([(2 * x + 1) / S - 1, -((2 * y + 1) / S - 1), np.ones_like(x)], -1)
    else:
        uv = np.stack([(x + 0.5) / S, (y + 0.5) / S], -1)
        if bnd == "zero":
            uv[:5] += 2.0  # outside the image
    uv = np.stack([uv, uv[::-1]]).astype(np.float32)
    tex = rng.random((1, 6, S, S, C) if bnd == "cube" else (1, S, S, C)).astype(np.float32)
    g = nonfinite(rng, rng.normal(size=(2, Hi, Wi, C)).astype(np.float32))
    kw = dict(filterMode=filt, boundaryMode=bnd)
    # (between two levels: of a level of weight zero no tap is added)
    da = np.full((2, Hi, Wi, 4), 1.3 / S, np.float32) if "mipmap" in filt else None
    t, u = dev(tex).requires_grad_(True), dev(uv).requires_grad_(uv_grad)
    DiffRast.texture(t, u, uvDA=None if da is None else dev(da), **kw).backward(dev(g))
    ref = O.texture_vjp(tex, uv, g, uvDA=da, **kw)[0]
    assert_same_nonfinite(host(t.grad), ref, "d_tex")


# texels that are not finite, also under weights of zero: outside the zero
# boundary's image, on the level a magnified surface does not use, and under
# footprints that fall on one texel
@pytest.mark.parametrize("filt", ["linear", "linear-mipmap-linear", "linear-mipmap-nearest"])
@pytest.mark.parametrize("bnd", ["wrap", "clamp", "zero"])
@pytest.mark.parametrize("lod", [1e-3, 1.3, 100.0])
def test_many_channels_nonfinite_texels(filt, bnd, lod):
    torch_dev()
    from diffrast import DiffRast
    rng = np.random.default_rng(5)
    Hi, Wi, Ht, Wt, C = 33, 40, 32, 64, 6
    uv, _ = smooth_uv(rng, 2, Hi, Wi, 0.9, 0.3, (0.0, 0.0))
    uv[:, -3:, -3:] = 4.0
    da = np.full((2, Hi, Wi, 4), lod / Wt, np.float32) * np.float32([1, 0.9, 0.4, 0.45])
    tex = rng.random((1, Ht, Wt, C)).astype(np.float32)
    tex[0, 0, 0, 1], tex[0, 20, 31, 2], tex[0, Ht - 1, Wt - 1, 4] = np.inf, np.nan, -np.inf
    g = rng.normal(size=(2, Hi, Wi, C)).astype(np.float32)
    kw = dict(filterMode=filt, boundaryMode=bnd)
    mip = "mipmap" in filt
    u = dev(uv).requires_grad_(True)
    out = DiffRast.texture(dev(tex), u, uvDA=dev(da) if mip else None, **kw)
    out.backward(dev(g))
    assert_same_nonfinite(host(out), O.texture(tex, uv, uvDA=da if mip else None, **kw), "out")
    ref = O.texture_vjp(tex, uv, g, uvDA=da if mip else None, **kw)[1]
    assert_same_nonfinite(host(u.grad), ref, "d_uv")


# a tile's d_tex terms are summed in fp64 from the first on: cotangents of
# +-2^26 that cancel within four pixels of a texel leave the small ones, which
# fp32 sums of a pixel row would lose (weights are 1, or 1/4 under a constant
# uv, so every product is exact)
@pytest.mark.parametrize("C", [1, 3, 4])
@pytest.mark.parametrize("kind", ["nearest", "nearest-constant", "cube", "wrap-constant"])
def test_sums_of_a_tile_are_exact(kind, C):
    torch_dev()
    from diffrast import DiffRast
    rng = np.random.default_rng(C)
    N, Hi, Wi, S = 2, 48, 64, 64
    y, x = np.meshgrid(np.arange(Hi) + 8, np.arange(Wi) // 4 + 8, indexing="ij")
    g = rng.integers(-3, 4, size=(N, Hi, Wi // 4, 4, C)).astype(np.float32) * 4
    at = rng.integers(0, 2, size=(N, Hi, Wi // 4, 1, C))
    np.put_along_axis(g, at, np.float32(2 ** 26), 3)
    np.put_along_axis(g, 2 + at, np.float32(-2 ** 26), 3)
    g = g.reshape(N, Hi, Wi, C)
    ref = np.zeros((S, S, C))
    if kind.startswith("nearest"):
        if kind == "nearest-constant":
            x, y = np.full_like(x, 5), np.full_like(y, 9)
        uv = np.stack([(x + 0.5) / S, (y + 0.5) / S], -1)
        kw = dict(filterMode="nearest", boundaryMode="wrap")
        np.add.at(ref, (y, x), g.astype(np.float64).sum(0))
    elif kind == "cube":
        uv = np.stack([(2 * x + 1) / S - 1, -((2 * y + 1) / S - 1), np.ones(x.shape)], -1)
        kw = dict(filterMode="linear", boundaryMode="cube")
        np.add.at(ref, (y, x), g.astype(np.float64).sum(0))
    else:  # the four corner texels
        uv = np.zeros((Hi, Wi, 2))
        kw = dict(filterMode="linear", boundaryMode="wrap")
        ref[np.ix_([0, S - 1], [0, S - 1])] = g.astype(np.float64).sum((0, 1, 2)) / 4
    uv = np.broadcast_to(uv, (N,) + uv.shape).astype(np.float32)
    shape = (1, 6, S, S, C) if kind == "cube" else (1, S, S, C)
    t = dev(rng.random(shape).astype(np.float32)).requires_grad_(True)
    DiffRast.texture(t, dev(uv), **kw).backward(dev(g))
    got = host(t.grad)[0]
    np.testing.assert_array_equal(got[4] if kind == "cube" else got, ref)


# the pyramid's backward on rows shorter and longer than a workgroup
@pytest.mark.parametrize("C", [1, 3, 4, 8])
@pytest.mark.parametrize("Ht,Wt", [(64, 2), (6, 2), (48, 16), (8, 520)])
@pytest.mark.parametrize("Nt", [1, 3])
def test_pyramid_backward_rows(C, Ht, Wt, Nt):
    torch_dev()
    rng = np.random.default_rng(Ht + Wt + C)
    uv = rng.uniform(0.0, 1.0, size=(3, 17, 19, 2)).astype(np.float32)
    da = rng.uniform(0.9, 1.1, size=(3, 17, 19, 4)).astype(np.float32) * np.float32(1.6 / max(Ht, Wt))
    tex = rng.random((Nt, Ht, Wt, C)).astype(np.float32)
    check(rng, tex, uv, da, "linear-mipmap-linear", "clamp")


def test_pyramid_of_more_rows_than_a_grid():
    """2^24 + 2 texel rows: as one workgroup of 256 threads a row, the
    pyramid's backward would be a grid of more than 2^32 threads, of which a
    launch runs a part (the general kernel's sides above 32,767 too)."""
    torch_dev()
    rng = np.random.default_rng(0)
    Ht, Wt = 2 ** 24 + 2, 2
    uv = rng.uniform(0.0, 1.0, size=(1, 16, 16, 2)).astype(np.float32)
    da = np.full((1, 16, 16, 4), 1.4 / Ht, np.float32)
    da[..., :2] = 0.0
    tex = rng.random((1, Ht, Wt, 1)).astype(np.float32)
    check(rng, tex, uv, da, "linear-mipmap-linear", "clamp")


def test_more_channels_than_a_tile_counts_in_32_bits():
    """2^25 + 5 channels: 256 pixels times chunks of four are more than 2^31
    items."""
    torch = torch_dev()
    from diffrast import DiffRast
    C = 2 ** 25 + 5
    tex = torch.rand(1, 1, 2, C, device="cuda")
    uv = torch.tensor([0.5, 0.5], device="cuda").reshape(1, 1, 1, 2)
    out = DiffRast.texture(tex, uv, filterMode="linear", boundaryMode="clamp").reshape(-1)
    assert float((out - tex[0, 0].mean(0)).abs().max()) < 1e-6


# a side above 32,767, where windows' 16-bit coordinates end: the general
# kernel at every compiled channel count, and the run-time one
@pytest.mark.parametrize("C", [1, 2, 3, 4, 6])
@pytest.mark.parametrize("filt,bnd", [("nearest", "wrap"), ("nearest", "zero"), ("linear", "clamp"),
                                      ("linear", "wrap"), ("linear-mipmap-linear", "zero"),
                                      ("linear-mipmap-nearest", "clamp")])
@pytest.mark.parametrize("Ht,Wt", [(2, 40000), (32768, 4)])
def test_long_sides(C, filt, bnd, Ht, Wt):
    torch_dev()
    rng = np.random.default_rng(C + Ht)
    uv = rng.uniform(-0.2, 1.2, size=(2, 18, 23, 2)).astype(np.float32)
    uv[:, 4:9] = uv[:, 4:5, :1]  # and pixels of one footprint
    da = rng.uniform(0.9, 1.1, size=(2, 18, 23, 4)).astype(np.float32)
    da *= np.float32([1.3 / Wt, 1.2 / Wt, 1.0 / Ht, 0.9 / Ht])
    tex = rng.random((1, Ht, Wt, C)).astype(np.float32)
    check(rng, tex, uv, da, filt, bnd)


# texel coordinates beyond 32 bits saturate, and the second one of a footprint
# wraps: every tap is inside the texture
@pytest.mark.parametrize("C", [1, 3, 4, 6])
@pytest.mark.parametrize("bnd", ["wrap", "clamp", "zero"])
@pytest.mark.parametrize("filt", ["nearest", "linear", "linear-mipmap-linear"])
def test_coordinates_beyond_32_bits(C, bnd, filt):
    torch_dev()
    from diffrast import DiffRast
    rng = np.random.default_rng(C)
    uv = rng.uniform(0.1, 0.9, size=(1, 9, 17, 2)).astype(np.float32)
    for k, value in enumerate([np.inf, -np.inf, np.nan, 5e7, -5e7, 3.4e7, 1e30]):
        uv[0, k, k + 2, k % 2] = value
        uv[0, k, k + 7] = value
    da = np.full((1, 9, 17, 4), 1.3 / 64, np.float32) if "mipmap" in filt else None
    tex = rng.random((1, 64, 64, C)).astype(np.float32)
    kw = dict(filterMode=filt, boundaryMode=bnd)
    t = dev(tex).requires_grad_(True)
    out = DiffRast.texture(t, dev(uv), uvDA=None if da is None else dev(da), **kw)
    assert_same_nonfinite(host(out), O.texture(tex, uv, uvDA=da, **kw), "out")
    g = rng.normal(size=out.shape).astype(np.float32)
    out.backward(dev(g))
    ref = O.texture_vjp(tex, uv, g, uvDA=da, **kw)[0]
    assert_same_nonfinite(host(t.grad), ref, "d_tex")


# uv that is not finite gives weights that are not: their products with
# cotangents of zero are NaN too
@pytest.mark.parametrize("C,bnd,filt", [(1, "wrap", "linear"), (3, "wrap", "linear"),
                                        (4, "wrap", "linear-mipmap-linear"), (3, "cube", "linear"),
                                        (6, "wrap", "linear"), (6, "clamp", "linear"),
                                        (6, "zero", "linear"), (6, "cube", "linear"),
                                        (6, "clamp", "linear-mipmap-linear"), (3, "wrap", "nearest"),
                                        (6, "zero", "nearest")])
@pytest.mark.parametrize("zero", ["all", "one"])
@pytest.mark.parametrize("uv_grad", [False, True])
def test_nonfinite_uv_zero_cotangent(C, bnd, filt, zero, uv_grad):
    torch_dev()
    from diffrast import DiffRast
    rng = np.random.default_rng(C)
    Hi, Wi, S = 33, 50, 64
    g = rng.normal(size=(2, Hi, Wi, C)).astype(np.float32)
    uv = rng.uniform(0.1, 0.9, size=(2, Hi, Wi, 3 if bnd == "cube" else 2)).astype(np.float32)
    for n, y, x, value in [(0, 3, 7, np.nan), (0, 20, 31, np.inf), (1, 9, 40, -np.inf), (1, 32, 49, np.nan)]:
        uv[n, y, x, 0] = value
        g[n, y, x, :C if zero == "all" else 1] = 0.0
    tex = rng.random((1, 6, S, S, C) if bnd == "cube" else (1, S, S, C)).astype(np.float32)
    kw = dict(filterMode=filt, boundaryMode=bnd)
    da = np.full((2, Hi, Wi, 4), 1.3 / S, np.float32) if "mipmap" in filt else None
    t, u = dev(tex).requires_grad_(True), dev(uv).requires_grad_(uv_grad)
    DiffRast.texture(t, u, uvDA=None if da is None else dev(da), **kw).backward(dev(g))
    ref = O.texture_vjp(tex, uv, g, uvDA=da, **kw)[0]
    assert_same_nonfinite(host(t.grad), ref, "d_tex")
