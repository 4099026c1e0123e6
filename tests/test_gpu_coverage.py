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
from rusterize_amd.device import BatchGraph, Context, DeviceBuffer, DeviceGeometry, Job, batch_rasterize, grid, \
    rasterize_device
from tests.test_gpu_parity import assert_same, degenerate_geometry, field_for, polygon_rings

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


def test_forced_masks_in_a_small_call(monkeypatch):
    # 10 polygons get no masks by themselves; RUSTERIZE_WIDE=always gives them
    # theirs (a context that never made a mask has no buffers for them), with
    # the same raster
    g = degenerate_geometry()
    field = field_for("float64", g.n_geoms, seed=3)
    info = grid(300, 200)
    ref = oracle.rasterize(g, oracle.copy_info(info), "float64", "sum", field=field, background=float("nan"))
    held = {}
    for wide in ("never", "always"):
        monkeypatch.setenv("RUSTERIZE_WIDE", wide)
        with Context(0) as ctx:
            dg, out = DeviceGeometry(ctx, g), DeviceBuffer(ctx, 200 * 300 * 8)
            d_field = DeviceBuffer.from_array(ctx, field)
            job = Job(dg, info, "float64", "sum", out, field=d_field, background=float("nan"))
            rasterize_device(ctx, job)
            ctx.synchronize()
            assert_same(job.result(), ref, f"wide {wide}")
            held[wide] = ctx.workspace_bytes()
            out.free()
            d_field.free()
            dg.free()
    assert held["always"] > held["never"]


def degenerate_rings(long):
    """The degenerate rings among 520 ordinary ones (so that the call takes
    masks); long: also rings of 400 vertices with one NaN, infinite or huge
    vertex each, and one left open."""
    rng = np.random.default_rng(5)
    d = degenerate_geometry()
    rings = [[d.xy[d.ring_vertex_offsets[r]:d.ring_vertex_offsets[r + 1]]
              for r in range(d.item_ring_offsets[i], d.item_ring_offsets[i + 1])] for i in range(d.n_geoms)]
    for k in range(520):
        p = rng.uniform(0, 300, (4, 2))
        rings.insert(int(rng.integers(0, len(rings))), [np.concatenate([p, p[:1]])])
    bad = [(np.nan, 90.0), (-np.nan, 60.0), (np.inf, 100.0), (-np.inf, 50.0), (1e300, 120.0), (120.0, np.nan),
           (150.0, -1e300), None]
    for k, v in enumerate(bad if long else []):
        a = np.linspace(0, 2 * np.pi, 401)
        p = np.stack([150 + (40 + 9 * k) * np.cos(a), 100 + (30 + 8 * k) * np.sin(a)], 1)
        p[400] = p[0]
        if v is None:
            p = p[:-3]
        else:
            p[97 + 30 * k] = v
        rings.insert(60 * k, [p])
    return polygon_rings(rings)


@pytest.mark.parametrize("binning,long", [("never", False), ("never", True), ("always", False), ("always", True)])
def test_degenerate_rings_in_masks(binning, long, monkeypatch):
    monkeypatch.setenv("RUSTERIZE_BINNING", binning)
    g = degenerate_rings(long)
    info = grid(300, 200)
    for dtype, fun, bg in (("float64", "sum", float("nan")), ("uint8", "count", 0), ("int32", "last", 0)):
        field = field_for(dtype, g.n_geoms, seed=7)
        got = _lib.rasterize(g, info, dtype, fun, field, None, None, 1, bg)
        ref = oracle.rasterize(g, oracle.copy_info(info), dtype, fun, field=field, background=bg)
        assert_same(got, ref, f"degenerate {dtype} {fun}")


def quads(n, size, long=False):
    """n quadrilaterals over most of size x size pixels; long: the first has
    400 vertices."""
    rng = np.random.default_rng(n + size)
    lo, hi = rng.uniform(-20, 0.08 * size, (n, 2)), rng.uniform(0.92 * size, size + 20, (n, 2))
    rings = []
    for k, ((x0, y0), (x1, y1)) in enumerate(zip(lo, hi)):
        p = np.array([(x0, y0), (x1, y0 + 7), (x1, y1), (x0 + 5, y1), (x0, y0)])
        if long and k == 0:
            p = np.concatenate([np.linspace(p[0], p[1], 397)[:-1], p[1:]])
        rings.append([p])
    return polygon_rings(rings)


@pytest.mark.parametrize("long", [False, True])
@pytest.mark.parametrize("dtype,fun,bg", [("float64", "sum", float("nan")), ("uint8", "count", 0),
                                          ("int16", "last", 0), ("int32", "max", 0)])
def test_masks_past_their_capacity(dtype, fun, bg, long, monkeypatch):
    # 600 items of about 240 mask blocks (128 bytes, 16 x 64 pixels each) on
    # 512 x 512 pixels: 148,000 blocks, where a scanned call holds at most
    # 2 bytes per pixel and 8 KiB per item: 42,496.  The items past that
    # compute their coverage from their edges, next to those with masks.
    monkeypatch.setenv("RUSTERIZE_BINNING", "never")
    g = quads(600, 512, long)
    field = field_for(dtype, g.n_geoms, seed=21)
    info = grid(512, 512)
    got = _lib.rasterize(g, info, dtype, fun, field, None, None, 1, bg)
    ref = oracle.rasterize(g, oracle.copy_info(info), dtype, fun, field=field, background=bg)
    assert_same(got, ref, f"past the mask capacity {dtype} {fun} {long}")


@pytest.mark.parametrize("binning,long,lines", [("never", False, 0), ("always", False, 0), ("always", True, 0),
                                                ("always", True, 60)])
def test_graph_replay_past_the_mask_capacity(binning, long, lines, monkeypatch):
    # 600 polygons captured while they are 16 x 16 pixels (2 mask blocks each)
    # and replayed grown to 62 x 62 in the same tiles (4 each): binned, the
    # capacity is the captured need + 64 = 1,264 of 2,400; scanned it is 64 per
    # item and more, so those grow to the whole raster.  60 lines of 79
    # segments beside them outgrow their bands in the same replay (4 entries
    # each where 2 were captured, with room for 64 more).
    monkeypatch.setenv("RUSTERIZE_BINNING", binning)
    rng = np.random.default_rng(8)
    centre = np.repeat(rng.uniform([32, 32], [96, 480], (600, 2)), 5, 0) // 64 * 64 + 32
    unit = np.tile([(-1, -1), (1, -0.9), (1, 1), (-0.9, 1), (-1, -1)], (600, 1))
    if long:  # the first ring has 400 vertices
        first = np.concatenate([np.linspace(unit[0], unit[1], 397)[:-1], unit[1:5]])
        unit, centre = np.concatenate([first, unit[5:]]), np.concatenate([centre[:1].repeat(400, 0), centre[5:]])
    nv = np.array([400 if long and k == 0 else 5 for k in range(600)] + [80] * lines)
    n = len(nv)
    kind = np.array([0] * 600 + [1] * lines, np.int32)

    def shape(half, tall):
        xy = [centre + half * unit]
        for k in range(lines):
            t = np.linspace(0, 1, 80)
            xy.append(np.stack([8 + 8 * k + 3 * np.sin(40 * t), 256.5 + tall * (t - 0.5)], 1))
        return Geometry(np.arange(n + 1), kind, np.arange(n + 1), np.concatenate([[0], np.cumsum(nv)]),
                        np.concatenate(xy))

    small, grown = shape(8.0, 12.0), shape(31.0 if binning == "always" else 1000.0, 62.0)
    info = grid(512, 512)
    field = field_for("float64", n, seed=5)
    with Context(0) as ctx:
        dg, out = DeviceGeometry(ctx, small), DeviceBuffer(ctx, 512 * 512 * 8)
        d_field = DeviceBuffer.from_array(ctx, field)
        job = Job(dg, info, "float64", "sum", out, field=d_field, background=float("nan"))
        graph = BatchGraph([job])
        try:
            for geom in (small, grown, grown, small):
                dg.set_xy(geom.xy)
                graph.launch()
                graph.synchronize()
                ref = oracle.rasterize(geom, oracle.copy_info(info), "float64", "sum", field=field,
                                       background=float("nan"))
                assert_same(job.result(), ref, "replay")
                rasterize_device(ctx, job)
                ctx.synchronize()
                assert_same(job.result(), ref, "eager between replays")
        finally:
            graph.close()
            out.free()
            d_field.free()
            dg.free()


def test_masks_of_a_large_raster_take_what_they_need(monkeypatch):
    # 600 quadrilaterals of 20 pixels on 8200 x 8200 (more pixels than masks are
    # reserved for unseen): at most 4 blocks of 128 bytes each, beside 2 bytes
    # per pixel (134 MB) if they were reserved by the raster's size
    monkeypatch.setenv("RUSTERIZE_BINNING", "never")
    n = 8200
    rng = np.random.default_rng(4)
    c = np.repeat(rng.uniform(40, n - 40, (600, 1, 2)), 5, 1)
    g = polygon_rings([[p] for p in c + 10 * np.array([(-1, -1), (1, -0.8), (1, 1), (-0.9, 1), (-1, -1)])])
    field = field_for("uint8", 600, seed=2)
    info = grid(n, n)
    with Context(0) as ctx:
        dg, out, d_field = DeviceGeometry(ctx, g), DeviceBuffer(ctx, n * n), DeviceBuffer.from_array(ctx, field)
        job = Job(dg, info, "uint8", "max", out, field=d_field)
        rasterize_device(ctx, job)
        ctx.synchronize()
        ref = oracle.rasterize(g, oracle.copy_info(info), "uint8", "max", field=field, background=0)
        assert_same(job.result(), ref, "600 small polygons on a large raster")
        assert ctx.workspace_bytes() < 16 << 20
        for b in (out, d_field, dg):
            b.free()


def test_masks_past_their_limit_when_the_need_is_known(monkeypatch):
    # the 600 quadrilaterals of test_masks_past_their_capacity in a batch whose
    # line bands make it read its totals: 148,000 blocks (19 MB) needed, of
    # which 42,000 and some (5.5 MB) are given
    monkeypatch.setenv("RUSTERIZE_BINNING", "never")
    t = np.linspace(0, 1, 80)
    lines = [np.stack([10 + 100 * t, 20 + 90 * t + 5 * np.sin(9 * t + k)], 1) for k in range(3)]
    sets = [quads(600, 512), Geometry(np.arange(4), np.ones(3, np.int32), np.arange(4), np.arange(4) * 80,
                                      np.concatenate(lines))]
    with Context(0) as ctx:
        jobs, refs, held = [], [], []
        for g, side, fun in zip(sets, (512, 128), ("sum", "count")):
            field = field_for("float64", g.n_geoms, seed=side)
            info = grid(side, side)
            dg, d_field = DeviceGeometry(ctx, g), DeviceBuffer.from_array(ctx, field)
            out = DeviceBuffer(ctx, side * side * 8)
            held += [dg, d_field, out]
            jobs.append(Job(dg, info, "float64", fun, out, field=d_field, background=float("nan")))
            refs.append(oracle.rasterize(g, oracle.copy_info(info), "float64", fun, field=field,
                                         background=float("nan")))
        for _ in range(2):
            batch_rasterize(ctx, jobs)
            ctx.synchronize()
            for job, ref in zip(jobs, refs):
                assert_same(job.result(), ref, job.fun)
        assert ctx.workspace_bytes() < 12 << 20
        for b in held:
            b.free()


@pytest.mark.parametrize("wide", [None, "never"])
@pytest.mark.parametrize("rows,cols", [(300, 400), (1500, 130)])
def test_long_rings_by_chunks(rows, cols, wide, monkeypatch):
    # rings on both sides of one, two and many chunks of 64 vertices, starting
    # anywhere in a chunk; smooth ones, whose chunks meet few rows, and ragged
    # ones, whose chunks meet most; with masks and computed strip by strip, in
    # a lone call and in a batch with a job before it
    if wide:
        monkeypatch.setenv("RUSTERIZE_WIDE", wide)
    rng = np.random.default_rng(rows)
    rings = []
    for k, nv in enumerate([5, 63, 64, 65, 128, 129, 130, 191, 320, 321, 4096, 4097, 4161, 9000]):
        for inner in (0.98, 0.2):
            a = np.sort(rng.uniform(0, 2 * np.pi, nv - 1))
            r = rng.uniform(inner, 1.0, nv - 1)
            p = np.stack([rng.uniform(0, cols) + cols * 0.6 * r * np.cos(a),
                          rng.uniform(0, rows) + rows * 0.6 * r * np.sin(a)], 1)
            rings.append([np.concatenate([p, p[:1]])])
            rings.append([np.array([(k, k), (k + 9, k), (k + 4, k + 7 + inner), (k, k)])[:3 + k % 2]])
    g = polygon_rings(rings)
    with Context(0) as ctx:
        dg = DeviceGeometry(ctx, g)
        held, jobs, refs = [dg], [], []
        for dtype, fun, bg in (("float64", "sum", float("nan")), ("uint8", "count", 0)):
            field = field_for(dtype, g.n_geoms, seed=cols)
            info = grid(cols, rows)
            out = DeviceBuffer(ctx, rows * cols * np.dtype(dtype).itemsize)
            d_field = DeviceBuffer.from_array(ctx, field)
            held += [out, d_field]
            jobs.append(Job(dg, info, dtype, fun, out, field=d_field, background=bg))
            refs.append(oracle.rasterize(g, oracle.copy_info(info), dtype, fun, field=field, background=bg))
            rasterize_device(ctx, jobs[-1])
            ctx.synchronize()
            assert_same(jobs[-1].result(), refs[-1], f"{dtype} {fun}")
        batch_rasterize(ctx, jobs[::-1])
        ctx.synchronize()
        for job, ref in zip(jobs, refs):
            assert_same(job.result(), ref, f"batch {job.dtype} {job.fun}")
        for b in held:
            b.free()


@pytest.mark.parametrize("binning", ["always", "never"])
@pytest.mark.parametrize("dtype", ["uint8", "int16", "float32", "float64"])
@pytest.mark.parametrize("rows,cols,n_layers", [(1, 1, 1), (15, 63, 1), (25, 65, 1), (65, 257, 1), (129, 1023, 2),
                                                (67, 130, 2100)])
def test_strips_without_masks(rows, cols, n_layers, dtype, binning, monkeypatch):
    # every item's coverage from its edges: units of 8 rows (a workgroup per
    # tile) and, with 2,100 layers, of 16; items in one, two and all of a
    # tile's 64-column words, past the raster on every side, and lines beside
    # them (the third kernel) in the last function
    monkeypatch.setenv("RUSTERIZE_BINNING", binning)
    monkeypatch.setenv("RUSTERIZE_WIDE", "never")
    g = polygons(rows, cols)
    info = _lib.raster_info(None, resolution=(1.0, 1.0), extent=(0, 0, cols, rows))
    for fun, bg in (("sum", 0), ("count", 2), ("first", 1), ("min", 0)):
        if fun == "min":
            t = np.linspace(0, 1, 40)
            line = np.stack([cols * t, rows * (0.5 + 0.4 * np.sin(9 * t))], 1)
            g = Geometry(np.arange(g.n_geoms + 2), np.append(g.item_kind, 1).astype(np.int32),
                         np.append(g.item_ring_offsets, g.item_ring_offsets[-1] + 1),
                         np.append(g.ring_vertex_offsets, g.ring_vertex_offsets[-1] + 40),
                         np.concatenate([g.xy, line]))
        layers = (np.arange(g.n_geoms) * 37 % n_layers // (3 if n_layers > 1 else 1)).astype(np.uint32)
        field = field_for(dtype, g.n_geoms, seed=rows + cols)
        got = _lib.rasterize(g, info, dtype, fun, field, None, layers, n_layers, bg)
        ref = oracle.rasterize(g, oracle.copy_info(info), dtype, fun, field=field, layer_of_geom=layers,
                               n_layers=n_layers, background=bg)
        assert_same(got, ref, f"{rows}x{cols}x{n_layers} {dtype} {fun} {binning}")


def wide_rings(rows, cols, top):
    """Rings of up to `top` vertices across the whole raster and past it, every
    second one open, and small ones at the words' edges."""
    rng = np.random.default_rng(cols)
    rings = []
    for k, nv in enumerate([4, 5, 63, 64, 300, 319, top, top]):
        a = np.sort(rng.uniform(0, 2 * np.pi, nv))
        r = rng.uniform(0.2, 1.0, nv)
        p = np.stack([cols * (0.5 + 0.6 * r * np.cos(a)), rows * (0.5 + 0.8 * r * np.sin(a))], 1)
        rings.append(p if k % 2 else np.concatenate([p, p[:1]]))
    for w in range(0, cols, 320):
        x, y = w + rng.uniform(-2, 2), rng.uniform(0, rows)
        rings.append(np.array([[x, y], [x + 70, y + 3], [x + 9, y + 20.5], [x, y]]))
    rvo = np.concatenate([[0], np.cumsum([len(r) for r in rings])])
    n = len(rings)
    return Geometry(np.arange(n + 1), np.zeros(n, np.int32), np.arange(n + 1), rvo, np.concatenate(rings))


@pytest.mark.parametrize("binning,top", [("never", 319), ("never", 900), ("always", 319), ("always", 900)])
@pytest.mark.parametrize("rows,cols", [(50, 26 * 64), (50, 26 * 64 + 1), (430, 64), (33, 238 * 64), (33, 238 * 64 + 1)])
def test_windows_across_wide_items(rows, cols, binning, top, monkeypatch):
    # items as wide as a wave's window (26 words of 64 columns; by rows 26
    # strips of one word) or a workgroup's (238), and one word wider: carries
    # from block to block, and the columns past a row's rightmost crossing
    # where open rings leave an odd count
    monkeypatch.setenv("RUSTERIZE_BINNING", binning)
    monkeypatch.setenv("RUSTERIZE_WIDE", "always")
    g = wide_rings(rows, cols, top)
    info = _lib.raster_info(None, resolution=(1.0, 1.0), extent=(0, 0, cols, rows))
    field = field_for("int32", g.n_geoms, seed=rows)
    for fun in ("sum", "last"):
        got = _lib.rasterize(g, info, "int32", fun, field, None, None, 1, 0)
        ref = oracle.rasterize(g, oracle.copy_info(info), "int32", fun, field=field, background=0)
        assert_same(got, ref, f"{rows}x{cols} {fun} {binning} {top}")


@pytest.mark.parametrize("res", [(0.25, 0.25), (32.0, 0.5), (2.0 ** -1005, 2.0 ** -1005), (0.3, 30.0), (1.0, 0.1)])
@pytest.mark.parametrize("binning", ["always", "never"])
def test_resolutions(res, binning, monkeypatch):
    # powers of two multiply by their exact reciprocal (far from the ends of
    # the range), all others divide; the third has coordinates near the
    # smallest normal numbers
    monkeypatch.setenv("RUSTERIZE_BINNING", binning)
    monkeypatch.setenv("RUSTERIZE_WIDE", "always")
    rows, cols = 130, 321
    g = polygons(rows, cols)
    scaled = Geometry(g.geom_item_offsets, g.item_kind, g.item_ring_offsets, g.ring_vertex_offsets, g.xy * np.array(res))
    info = _lib.raster_info(None, resolution=res, extent=(0, 0, cols * res[0], rows * res[1]))
    field = field_for("float64", g.n_geoms, seed=5)
    got = _lib.rasterize(scaled, info, "float64", "sum", field, None, None, 1, float("nan"))
    ref = oracle.rasterize(scaled, oracle.copy_info(info), "float64", "sum", field=field, background=float("nan"))
    assert_same(got, ref, f"{res} {binning}")
