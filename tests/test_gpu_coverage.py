"""GPU parity of the coverage masks and of the kernels that fold them, bit for
bit against the oracle, at the sizes where they can go wrong: outputs whose
width is one off a mask word (64 columns), a tile or a 64-byte line, heights
one off a strip (16 rows) or a tile; items of one edge chunk, more, and more
than a wave's (320 vertices); boxes of one wave window and of many; rings
left open; more than 64 items over one strip; launches with a workgroup per
tile and, with enough layers, with a wave per strip; items from one launch
(k_items) and from the list kernels."""
import numpy as np
import pytest

from oracle import oracle
from rusterize_amd import _lib
from rusterize_amd._lib import Geometry
from tests.test_gpu_parity import assert_same, field_for

pytestmark = pytest.mark.gpu


def polygons(rows, cols):
    """Rings of 3 to 700 vertices from a fraction of a pixel to past the raster."""
    rng = np.random.default_rng(rows * 1000 + cols)
    rings = []
    top = 700 if cols > 200 else 319  # (at most 320 with the closing vertex: one launch covers all)
    for k, nv in enumerate([3, 4, 5, 16, 63, 64, 65, 128, 319, 320, 321, 700] * 4 + [5] * 80):
        cx, cy = rng.uniform(-5, cols + 5), rng.uniform(-5, rows + 5)
        size = (0.4, 3.0, 20.0, 1.2 * max(rows, cols))[k % 4] if k < 48 else 30.0
        nv = min(nv, top)
        a = np.sort(rng.uniform(0, 2 * np.pi, nv))
        r = size * rng.uniform(0.3, 1.0, nv)
        p = np.stack([cx + r * np.cos(a), cy + r * np.sin(a)], 1)
        rings.append(p if k % 7 == 6 else np.concatenate([p, p[:1]]))  # every seventh ring is open
    n = len(rings)
    rvo = np.concatenate([[0], np.cumsum([len(r) for r in rings])])
    return Geometry(np.arange(n + 1), np.zeros(n, np.int32), np.arange(n + 1), rvo, np.concatenate(rings))


@pytest.mark.parametrize("binning", ["always", "never"])
@pytest.mark.parametrize("dtype", ["uint8", "int16", "float32", "float64"])
@pytest.mark.parametrize("rows,cols,n_layers", [(1, 1, 1), (15, 63, 1), (64, 64, 1), (65, 257, 1), (129, 1023, 3),
                                                (130, 321, 0), (67, 130, 2100)])
def test_coverage_sizes(rows, cols, n_layers, dtype, binning, monkeypatch):
    monkeypatch.setenv("RUSTERIZE_BINNING", binning)
    if n_layers == 0:  # more than 12,288 tiles for every tile width
        n_layers = 2100 if np.dtype(dtype).itemsize <= 2 else 700
    g = polygons(rows, cols)
    info = _lib.raster_info(None, resolution=(1.0, 1.0), extent=(0, 0, cols, rows))
    layers = (np.arange(g.n_geoms) * 37 % n_layers // (3 if n_layers > 1 else 1)).astype(np.uint32)
    field = field_for(dtype, g.n_geoms, seed=rows + cols)
    for fun, bg in (("sum", 0), ("count", 2), ("last", 1), ("max", 0)):
        got = _lib.rasterize(g, info, dtype, fun, field, None, layers, n_layers, bg)
        ref = oracle.rasterize(g, oracle.copy_info(info), dtype, fun, field=field, layer_of_geom=layers,
                               n_layers=n_layers, background=bg)
        assert_same(got, ref, f"{rows}x{cols}x{n_layers} {dtype} {fun} {binning}")
