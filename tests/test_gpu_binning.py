"""Tile binning at the sizes where its path changes, against the CPU oracle:
remainders of the four-tile steps, the 64 KiB of LDS that need no extra
attribute (16,384 tiles), the most tiles its LDS counters hold (40,000) and
one more (the counters in memory)."""
import numpy as np
import pytest

import oracle as O
from parity import dev, host, torch_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tiles", [1, 2, 5, 16384, 16385, 39999, 40000, 40001])
def test_tile_counts(tiles):
    torch_dev()
    from diffrast import DiffRast
    rng = np.random.default_rng(tiles)
    H, W, T = 16, 16 * tiles - 3, 1500
    half = 3e-3 if tiles > 100 else 0.5
    xyz = rng.uniform(-1.1, 1.1, size=(1, 3 * T, 3)).astype(np.float32)
    xyz[..., 0] = np.repeat(rng.uniform(-1.0, 1.0, size=(1, T)), 3, axis=1) + \
        rng.uniform(-half, half, size=(1, 3 * T))
    pos = np.concatenate([xyz, np.ones((1, 3 * T, 1), np.float32)], 2).astype(np.float32)
    tri = np.arange(3 * T, dtype=np.int32).reshape(T, 3)
    counts = host(DiffRast.rasterizeTileCounts(dev(pos), dev(tri), (H, W)))
    np.testing.assert_array_equal(counts, O.rasterize_tile_counts(pos, tri, (H, W)))
    r, db = DiffRast.rasterize(dev(pos), dev(tri), (H, W))
    r, db = DiffRast.rasterize(dev(pos), dev(tri), (H, W))  # lists sized by the first call
    rr, rdb = O.rasterize(pos, tri, (H, W), max_per_tile=0)
    np.testing.assert_array_equal(host(r), rr)
    np.testing.assert_array_equal(host(db), rdb)


def test_large_image_under_capture():
    """More than 64 KiB of LDS counters inside a HIP graph: every replay, with
    eager work between them, gives the eager result."""
    torch = torch_dev()
    from diffrast import DiffRast
    rng = np.random.default_rng(3)
    H, W, T = 2080, 2081, 900
    xyz = np.repeat(rng.uniform(-1, 1, size=(1, T, 3)), 3, axis=1) + \
        rng.uniform(-0.05, 0.05, size=(1, 3 * T, 3))
    pos = dev(np.concatenate([xyz, np.ones((1, 3 * T, 1))], 2).astype(np.float32))
    tri = dev(np.arange(3 * T, dtype=np.int32).reshape(T, 3))
    other = dev((xyz * 0.5).astype(np.float32))
    other = torch.cat([other, torch.ones_like(other[..., :1])], -1).contiguous()
    ref = host(DiffRast.rasterize(pos, tri, (H, W))[0])
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        for _ in range(2):
            DiffRast.rasterize(pos, tri, (H, W))
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            out, _ = DiffRast.rasterize(pos, tri, (H, W))
        for _ in range(3):
            out.zero_()
            DiffRast.rasterize(other, tri, (H, W))
            g.replay()
            torch.cuda.synchronize()
            np.testing.assert_array_equal(host(out), ref)
