"""The ops as autograd nodes: what a Python autograd function over the same
calls did with hooks on saved tensors, in-place changes, transforms, partial
and missing cotangents, and other threads and streams."""
import threading

import numpy as np
import pytest

import scenes
from parity import dev, host, torch_dev

pytestmark = pytest.mark.gpu


def scene():
    sc = scenes.textured_icosphere(N=2, H=40, W=36, level=2, tex_size=16)
    return dev(sc["pos"]), dev(sc["tri"]), dev(sc["uv"]), dev(sc["tex"])


def chain(pos, tri, uv, tex):
    from diffrast import DiffRast
    rast, db = DiffRast.rasterize(pos, tri, (40, 36))
    a, da = DiffRast.interpolate(uv, rast, tri, rastDB=db, diffAttrs=[0, 1])
    col = DiffRast.texture(tex, a, uvDA=da, filterMode="linear-mipmap-linear", boundaryMode="clamp")
    return DiffRast.antialias(col, rast, pos, tri)


def test_saved_tensor_hooks_are_called():
    torch = torch_dev()
    pos, tri, uv, tex = scene()
    pos.requires_grad_(True)
    ref = torch.autograd.grad(chain(pos, tri, uv, tex).square().sum(), pos)[0]
    seen = [0, 0]

    def pack(t):
        seen[0] += 1
        return t.cpu()

    def unpack(t):
        seen[1] += 1
        return t.cuda()
    with torch.autograd.graph.saved_tensors_hooks(pack, unpack):
        out = chain(pos, tri, uv, tex).square().sum()
    got = torch.autograd.grad(out, pos)[0]
    assert seen[0] >= 15 and seen[1] >= 15
    np.testing.assert_allclose(host(got), host(ref), rtol=1e-5, atol=1e-5 * float(ref.abs().max()))


def test_in_place_change_is_refused():
    torch = torch_dev()
    pos, tri, uv, tex = scene()
    uv2 = uv.requires_grad_(True).clone()
    out = chain(pos, tri, uv2, tex)
    uv2.add_(1.0)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        out.sum().backward()


def test_transforms_are_refused():
    """vmap, functorch's gradients and forward mode pass autograd nodes by:
    each op refuses them by name (and takes the same call without)."""
    torch = torch_dev()
    from diffrast import DiffRast
    from diffrast.fit import mse_loss
    import torch.autograd.forward_ad as forward_ad
    pos, tri, uv, tex = scene()
    rast, db = DiffRast.rasterize(pos, tri, (8, 8))
    a, _ = DiffRast.interpolate(uv, rast, tri)
    col = DiffRast.texture(tex, a)
    topo = DiffRast.antialiasConstructTopologyHash(tri)
    ops = [(lambda t: DiffRast.rasterize(t, tri, (8, 8))[0], pos),
           (lambda t: DiffRast.interpolate(t, rast, tri)[0], uv),
           (lambda t: DiffRast.texture(t, a), tex),
           (lambda t: DiffRast.antialias(t, rast, pos, tri, topologyHash=topo), col),
           (lambda t: mse_loss(t, col), col.clone())]
    for op, x in ops:
        assert torch.isfinite(op(x)).all()
        for call in (lambda: torch.func.vmap(op)(x[None]),
                     lambda: torch.func.grad(lambda t: op(t).sum())(x),
                     lambda: torch.func.jvp(op, (x,), (x,))):
            with pytest.raises(RuntimeError, match="torch::autograd::Function with functorch"):
                call()
        with forward_ad.dual_level():
            with pytest.raises(RuntimeError, match="jvp is not implemented"):
                op(forward_ad.make_dual(x, x))


def test_partial_cotangents():
    """Only one of an op's outputs used; a leaf that gets no gradient."""
    torch = torch_dev()
    from diffrast import DiffRast
    pos, tri, uv, tex = scene()
    pos.requires_grad_(True), uv.requires_grad_(True)
    rast, db = DiffRast.rasterize(pos, tri, (40, 36))
    g = torch.randn_like(rast)
    one = torch.autograd.grad(rast, pos, g, retain_graph=True)[0]
    both = torch.autograd.grad([rast, db], pos, [g, torch.zeros_like(db)], retain_graph=True)[0]
    np.testing.assert_array_equal(host(one), host(both))
    only_db = torch.autograd.grad(db, pos, torch.ones_like(db), retain_graph=True)[0]
    assert torch.isfinite(only_db).all()
    a, da = DiffRast.interpolate(uv, rast.detach(), tri, rastDB=db.detach(), diffAttrs="all")
    da_only = torch.autograd.grad(da, uv, torch.ones_like(da), retain_graph=True)[0]
    ref = torch.autograd.grad([a, da], uv, [torch.zeros_like(a), torch.ones_like(da)])[0]
    np.testing.assert_allclose(host(da_only), host(ref), rtol=1e-5, atol=1e-4)


def test_threads_and_streams():
    """Each thread on its own stream, forward and backward, repeatedly: the
    results of one thread alone."""
    torch = torch_dev()
    pos, tri, uv, tex = scene()

    def step(p):
        p = p.detach().clone().requires_grad_(True)
        return torch.autograd.grad(chain(p, tri, uv, tex).square().sum(), p)[0]
    inputs = [pos * (1 + 0.01 * i) for i in range(3)]
    refs = [host(step(p)) for p in inputs]
    torch.cuda.synchronize()
    bad = []

    def work(i):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(5):
                    got = host(step(inputs[i]))
                    np.testing.assert_allclose(got, refs[i], rtol=1e-4,
                                               atol=1e-4 * np.abs(refs[i]).max())
        except Exception as e:  # reported by the main thread
            bad.append(e)
    ts = [threading.Thread(target=work, args=(i,)) for i in range(3)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not bad, bad[0]


def test_side_inputs_are_checked():
    """Inputs beside the main ones that are on the host, or too small for
    what the kernels read of them, are ValueErrors before any launch."""
    torch = torch_dev()
    from diffrast import DiffRast
    pos, tri, uv, tex = scene()
    rast, db = DiffRast.rasterize(pos, tri, (40, 36))
    a, da = DiffRast.interpolate(uv, rast, tri, rastDB=db, diffAttrs="all")
    mip = dict(filterMode="linear-mipmap-linear")
    d = torch.nn.functional.pad(a, (0, 1), value=1.0)
    cube = torch.rand(1, 6, 8, 8, 3, device="cuda")
    bias = torch.zeros(a.shape[:3])
    for call, msg in [
            (lambda: DiffRast.interpolate(uv, rast, tri, rastDB=db.cpu(), diffAttrs="all"), "rastDB"),
            (lambda: DiffRast.interpolate(uv, rast, tri, rastDB=db.cpu(), diffAttrs=[0]), "rastDB"),
            (lambda: DiffRast.texture(tex, a, uvDA=da.cpu(), **mip), "uvDA"),
            (lambda: DiffRast.texture(tex, a, uvDA=da, mipLevelBiasMap=bias, **mip), "mipLevelBiasMap"),
            (lambda: DiffRast.texture(cube, d, uvDA=torch.zeros(*a.shape[:3], 6), boundaryMode="cube",
                                      **mip), "uvDA")]:
        with pytest.raises(ValueError, match=msg + " must be on the device"):
            call()
    col = DiffRast.texture(tex, a)
    with pytest.raises(ValueError, match="color's batch"):
        DiffRast.antialias(col, rast, pos[:1], tri)
    with pytest.raises(ValueError, match="topologyHash must be"):
        DiffRast.antialias(col, rast, pos, tri, topologyHash=tri[:4])
    topo = DiffRast.antialiasConstructTopologyHash(tri)
    out = DiffRast.antialias(col, rast, pos, tri, topologyHash=topo)
    np.testing.assert_array_equal(host(out), host(DiffRast.antialias(col, rast, pos, tri)))


def test_saved_pos_back_at_another_tensors_address():
    """The backward of a forward whose saved pos a hook brings back in new
    memory, at the address of the last forward's pos by then freed: it must
    not take that forward's per-triangle values for its own."""
    torch = torch_dev()
    from diffrast import DiffRast
    rng = np.random.default_rng(3)
    V, T = 1_000_000, 40  # 16 MB: a block of the allocator's own
    tri = dev(np.arange(3 * T, dtype=np.int32).reshape(T, 3))

    def vertices():
        p = rng.uniform(-1, 1, size=(1, V, 4)).astype(np.float32)
        p[..., 3] = 1.0
        return dev(p)
    a, b = vertices().requires_grad_(True), vertices()
    g = torch.randn(1, 64, 64, 4, device="cuda")
    at = {}

    def pack(t):
        return t.cpu() if t.shape == a.shape else t.detach()

    def unpack(t):
        if t.is_cuda:
            return t
        t = t.cuda()
        at["unpacked"] = t.data_ptr()
        return t
    ref = torch.autograd.grad(DiffRast.rasterize(a * 1.0, tri, (64, 64))[0], a, g)[0]
    torch.cuda.synchronize()
    with torch.autograd.graph.saved_tensors_hooks(pack, unpack):
        rast = DiffRast.rasterize(a * 1.0, tri, (64, 64))[0]
    with torch.no_grad():
        other = b * 1.0
        at["other"] = other.data_ptr()
        DiffRast.rasterize(other, tri, (64, 64))
        del other
    got = torch.autograd.grad(rast, a, g)[0]
    assert at["unpacked"] == at["other"]  # the case that is meant
    np.testing.assert_array_equal(host(got), host(ref))
