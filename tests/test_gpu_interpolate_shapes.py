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
