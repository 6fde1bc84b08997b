"""The map build's tiles of 4 x 4 x 4 points per 3 A cell: spacings that give
a cell 3, 8, 9 or 13 points an axis, boxes that cut cells, receptors whose
lists need more than one LDS part, and type counts at the row widths (4, 8,
16).  FP64 maps equal the oracle's bit for bit; the cells' prefix sums equal
a host count (through the maps)."""
import numpy as np
import pytest

import pyoracle as po
import smina_gpu as sg
from common import receptor

pytestmark = pytest.mark.gpu


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
    ctx = sg.Context(0)
    n, smooth, fast = sg.build_tables(sf)
    ctx.upload_tables(n, smooth, fast)
    rid = ctx.upload_receptor(rec.xyz, rec.type)
    gid = ctx.build_grids(rid, gd, types, sg.FP64)
    for t in types:
        assert np.array_equal(ctx.download_grid(gid, t, gd), o.grid(t)), t
    ctx.close()
