"""interpolate for any attribute count and any set of derivatives, against
the CPU oracle: chunks of four attributes with every remainder, derivative
indices out of order, repeated, and spread over chunks, as many as travel with
the launch (32) and more; tiles with more
vertex rows than the backward's table holds."""
import numpy as np
import pytest

import oracle as O
import scenes
from parity import assert_fwd_close, assert_grad_close, dev, host, torch_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("A,diff", [(1, None), (1, "all"), (4, "all"), (4, [3]), (5, None),
                                    (5, [0, 1]), (6, "all"), (7, [6, 0, 6]), (8, [0, 1]),
                                    (9, [8, 4, 3, 0]), (16, "all"), (17, None), (33, [32, 1]),
                                    (40, list(range(32))), (40, list(range(39, 5, -1)))])
@pytest.mark.parametrize("shared", [True, False])
@pytest.mark.parametrize("level,H,W", [(2, 50, 41), (6, 33, 64)])  # level 6: ~8 triangles a pixel
def test_any_shape(A, diff, shared, level, H, W):
    torch_dev()
    from diffrast import DiffRast
    sc = scenes.textured_icosphere(N=2, H=H, W=W, level=level, tex_size=8)
    rng = np.random.default_rng(A)
    V = sc["pos"].shape[1]
    attr = rng.normal(size=(V, A) if shared else (2, V, A)).astype(np.float32)
    rast, db = O.rasterize(sc["pos"], sc["tri"], (H, W), max_per_tile=0)
    kw = dict(rastDB=db, diffAttrs=diff) if diff else {}
    ref, ref_da = O.interpolate(attr, rast, sc["tri"], **kw)
    a, r, d = dev(attr).requires_grad_(True), dev(rast).requires_grad_(True), dev(db).requires_grad_(True)
    out, da = DiffRast.interpolate(a, r, dev(sc["tri"]), **(dict(rastDB=d, diffAttrs=diff) if diff else {}))
    assert_fwd_close(host(out), ref)
    g = rng.normal(size=ref.shape).astype(np.float32)
    if diff:
        assert_fwd_close(host(da), ref_da)
        gda = rng.normal(size=ref_da.shape).astype(np.float32)
        import torch
        torch.autograd.backward([out, da], [dev(g), dev(gda)])
        d_attr, d_rast, d_db = O.interpolate_vjp(attr, rast, sc["tri"], g, d_out_da=gda, **kw)
        assert_grad_close(host(d.grad), d_db, "d_rast_db", rtol=1e-5)
    else:
        out.backward(dev(g))
        d_attr, d_rast, _ = O.interpolate_vjp(attr, rast, sc["tri"], g)
    assert_grad_close(host(r.grad), d_rast, "d_rast", rtol=1e-5)
    assert_grad_close(host(a.grad), d_attr, "d_attr")


@pytest.mark.parametrize("A,diff", [(1, None), (5, None), (8, [0, 1]), (6, "all"), (1, "all")])
def test_sums_of_a_tile_are_exact(A, diff):
    """A tile's d_attr terms are summed in fp64: cotangents of +-2^26 that
    cancel within a pixel row leave the ones between them, which fp32 sums of
    the row would lose.  One triangle everywhere at u = v = 0, so vertex 0
    takes every cotangent whole and the derivatives' u terms (db = (1, 0, 0,
    0)) go to vertices 0 and 1."""
    torch = torch_dev()
    from diffrast import DiffRast
    rng = np.random.default_rng(A)
    N, H, W = 1, 64, 80
    rast = np.zeros((N, H, W, 4), np.float32)
    rast[..., 3] = 1.0
    db = np.zeros_like(rast)
    db[..., 0] = 1.0

    def cotangent(n):
        g = rng.integers(-3, 4, size=(N, H, W, n)).astype(np.float32)
        at = rng.integers(0, 8, size=(N, H, W // 16, n))
        big = g.reshape(N, H, W // 16, 16, n)
        np.put_along_axis(big, at[:, :, :, None], np.float32(2 ** 26), 3)
        np.put_along_axis(big, 8 + at[:, :, :, None], np.float32(-2 ** 26), 3)
        return g
    attr = dev(rng.normal(size=(1, 3, A)).astype(np.float32)).requires_grad_(True)
    tri = dev(np.array([[0, 1, 2]], np.int32))
    g = cotangent(A)
    ref = np.zeros((3, A))
    ref[0] = g.astype(np.float64).sum((0, 1, 2))
    if diff is None:
        out, _ = DiffRast.interpolate(attr, dev(rast), tri)
        out.backward(dev(g))
    else:
        idx = list(range(A)) if diff == "all" else diff
        gda = cotangent(2 * len(idx))
        out, da = DiffRast.interpolate(attr, dev(rast), tri, rastDB=dev(db), diffAttrs=diff)
        torch.autograd.backward([out, da], [dev(g), dev(gda)])
        u_term = gda[..., 0::2].astype(np.float64).sum((0, 1, 2))
        ref[0, idx] -= u_term
        ref[1, idx] += u_term
    np.testing.assert_array_equal(host(attr.grad)[0], ref)


def test_more_attributes_than_a_tile_counts_in_32_bits():
    """2^25 + 5 attributes: the forward's 256 pixels times chunks of four are
    more than 2^31 items."""
    torch = torch_dev()
    from diffrast import DiffRast
    A = 2 ** 25 + 5
    attr = torch.rand(1, 3, A, device="cuda")
    rast = torch.tensor([0.25, 0.5, 0.0, 1.0], device="cuda").reshape(1, 1, 1, 4)
    tri = torch.tensor([[0, 1, 2]], dtype=torch.int32, device="cuda")
    out = DiffRast.interpolate(attr, rast, tri)[0].reshape(-1)
    want = 0.25 * attr[0, 0] + 0.25 * attr[0, 1] + 0.5 * attr[0, 2]
    assert float((out - want).abs().max()) < 1e-6
