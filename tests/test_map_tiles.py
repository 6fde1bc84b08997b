"""The map build's tiles of 4 x 4 x 4 points per 3 A cell: spacings that give
a cell 3, 8, 9 or 13 points an axis, boxes that cut cells, type counts at the
row widths (4, 8, 16), cells whose lists are one LDS part (512 records), one
entry more, and three parts, and cells with more tiles than the launch has
waves for one (each then takes its parts again for the next tiles).  FP64 maps
equal the oracle's bit for bit with each kind of table; the cells' prefix sums
equal a host count (through the maps)."""
import numpy as np
import pytest

import pyoracle as po
import smina_gpu as sg
from common import receptor

pytestmark = pytest.mark.gpu


def context(sf, kind):
    ctx = sg.Context(0)
    n, smooth, fast = sg.build_tables(sf)
    _, qs, qf = sg.build_qtables(sf)
    ctx.upload_tables(n, smooth, fast, qsmooth=qs, qfast=qf)
    if kind == "spline":
        ctx.upload_splines(*sg.build_splines(sf, 10.0))
    return ctx


@pytest.mark.parametrize("center,size,spacing,ntypes,nheavy", [
    ((0.0, 0.0, 0.0), (9.0, 6.0, 12.0), 0.375, 4, 1800),
    ((0.4, -1.3, 2.2), (7.1, 10.3, 5.5), 0.375, 5, 1800),
    ((0.1, 0.2, 0.3), (6.0, 6.0, 6.0), 1.1, 8, 1800),
    ((0.1, 0.2, 0.3), (4.0, 4.0, 4.0), 0.23, 9, 1800),
    ((5.0, 5.0, 5.0), (6.0, 6.0, 6.0), 0.375, 12, 6000),
])
def test_maps_match_oracle(center, size, spacing, ntypes, nheavy):
    rec = receptor(3, nheavy) if nheavy != 1800 else receptor()
    gd = sg.grid_dims(center, size, spacing)
    sf = sg.vina_scoring()
    types = list(range(2, 2 + ntypes))
    o = po.Oracle(sf, rec.xyz, rec.type, gd)
    o.build_grids(types)
    ctx = context(sf, "linear")
    rid = ctx.upload_receptor(rec.xyz, rec.type)
    gid = ctx.build_grids(rid, gd, types, sg.FP64)
    for t in types:
        assert np.array_equal(ctx.download_grid(gid, t, gd), o.grid(t)), t
    ctx.close()


def dense_receptor(nheavy, center):
    """heavy atoms within 4 A of the centre, and a hydrogen after every 7th:
    the one cell of a box of less than 3 A around it lists every heavy atom"""
    rng = np.random.default_rng(nheavy)
    n = nheavy + nheavy // 7
    v = rng.standard_normal((n, 3))
    xyz = np.asarray(center) + 4.0 * rng.uniform(0, 1, (n, 1)) ** (1 / 3) * v / np.linalg.norm(v, axis=1)[:, None]
    types = rng.integers(2, 15, n).astype(np.int32)
    types[np.arange(nheavy // 7) * 8 + 7] = 1
    assert np.sum(types > 1) == nheavy
    return xyz, types, rng.uniform(-0.5, 0.5, n)


def longest_list(xyz, types, gd):
    """the entries of the fullest cell: heavy atoms within the cutoff of the
    box and of the cell's brick, from the first probe coordinate in it"""
    axes = []
    for d in range(3):
        p = gd.begin[d] + np.arange(gd.n[d] + 1) * ((gd.end[d] - gd.begin[d]) / gd.n[d])
        axes.append(sorted({(np.floor(p[np.floor(p / 3) == c][0] / 3) * 3, np.ceil(p[np.floor(p / 3) == c][0] / 3) * 3)
                            for c in np.unique(np.floor(p / 3))}))
    heavy = xyz[types > 1]
    lo, hi = np.array(gd.begin[:3]), np.array(gd.end[:3])

    def near(lo, hi):
        return np.sum((np.clip(heavy, lo, hi) - heavy) ** 2, axis=1) < 64.0
    return max(int(np.sum(near(lo, hi) & near(np.array([a[0], b[0], c[0]]), np.array([a[1], b[1], c[1]]))))
               for a in axes[0] for b in axes[1] for c in axes[2])


@pytest.mark.parametrize("kind", ["linear", "spline", "charged"])
@pytest.mark.parametrize("nheavy,size,spacing", [
    (512, 2.4, 0.3), (513, 2.4, 0.3), (1100, 2.4, 0.3),
    (600, 2.6, 0.063),  # 43 points an axis: 1,331 tiles a cell
])
def test_lists_past_one_part(nheavy, size, spacing, kind):
    center = (1.5, 1.5, 1.5)
    xyz, types, q = dense_receptor(nheavy, center)
    gd = sg.grid_dims(center, (size,) * 3, spacing)
    assert longest_list(xyz, types, gd) == nheavy
    sf = sg.builtin_scoring("ad4_scoring") if kind == "charged" else sg.vina_scoring()
    q = q if kind == "charged" else None
    o = po.Oracle(sf, xyz, types, gd, receptor_charges=q)
    if kind == "spline":
        o.use_splines(10.0)
    want = [2, 7, 13] if spacing > 0.1 else [7]
    o.build_grids(want)
    ctx = context(sf, kind)
    rid = ctx.upload_receptor(xyz, types, charges=q)
    gid = ctx.build_grids(rid, gd, want, sg.FP64)
    for t in want:
        assert np.array_equal(ctx.download_grid(gid, t, gd), o.grid(t)), t
        if kind == "charged":
            assert np.array_equal(ctx.download_grid(gid, t, gd, charge=True), o.charge_grid(t)), t
    ctx.close()


def test_few_cells_of_many_points_fill_the_device():
    """1.77 million points as 64 cells of a 6 A box take no more than 3 times
    what they take as 1,000 cells of a 24 A box (2.1 ms; the 6 A box 1.0 ms,
    and 56 ms with a workgroup per cell)"""
    rec = receptor()
    ctx = context(sg.vina_scoring(), "spline")
    rid = ctx.upload_receptor(rec.xyz, rec.type)
    ms = {}
    for size, spacing in ((24.0, 0.2), (6.0, 0.05)):
        gd = sg.grid_dims((0.0, 0.0, 0.0), (size,) * 3, spacing)
        times = []
        for _ in range(4):
            gid = ctx.build_grids(rid, gd, [2, 7, 8, 13], sg.FP32)
            times.append(ctx.last_ms("grid_build"))
            ctx.check(sg.lib.sgpu_release_grid(ctx.h, gid))
        ms[size] = min(times)
    ctx.close()
    print(ms, flush=True)
    assert ms[6.0] < 3 * ms[24.0], ms
