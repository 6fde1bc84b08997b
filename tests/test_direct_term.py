"""The direct receptor term's lists, read in batches of 4 records: receptors
whose lists have fewer entries than a batch, a whole number of batches, and
one more or less.  FP64 equals the oracle bit for bit on both table forms
(evaluation and final rescoring); FP32 is within the reference's bound for
an evaluation away from a discontinuity (1e-3 relative)."""
import numpy as np
import pytest

import pyoracle as po
import smina_gpu as sg
from common import gd_c0, ligand, receptor

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("approx", ["linear", "spline"])
@pytest.mark.parametrize("natoms", [1, 3, 4, 5, 8, 9, 41])
def test_lists_around_the_batch_size(natoms, approx):
    rec, lig, gd, sf = receptor(), ligand(), gd_c0(), sg.vina_scoring()
    near = np.argsort(np.linalg.norm(rec.xyz, axis=1) + 100.0 * (rec.type <= 1))[:natoms]
    xyz, types = rec.xyz[near], rec.type[near]
    o = po.Oracle(sf, xyz, types, gd)
    ctx = sg.Context(0)
    n, smooth, fast = sg.build_tables(sf)
    ctx.upload_tables(n, smooth, fast)
    if approx == "spline":
        o.use_splines(10.0)
        ctx.upload_splines(*sg.build_splines(sf, 10.0))
    m = o.add_model(lig.desc_ptr)
    f = sg.Flat(lig)
    rid = ctx.upload_receptor(xyz, types)
    rng = np.random.default_rng(natoms)
    confs = np.repeat(f.initial_conf()[None], 12, 0)
    confs[:, :3] += rng.uniform(-4.0, 4.0, (12, 3))
    for prec in (sg.FP64, sg.FP32):
        bid = ctx.upload_models([f], prec)
        e, g, _ = ctx.eval_confs(bid, [0] * 12, confs, f.change_size, f.natoms, (10.0,) * 3, receptor_id=rid, gd=gd,
                                 slope=10.0)
        s = ctx.score(bid, rid, gd, [0] * 12, confs, 0)
        for k in range(12):
            eo, go, _ = o.eval_deriv(m, confs[k], (10.0,) * 3, backend=1, slope=10.0)
            assert s[k] == o.eval(m, confs[k])
            if prec == sg.FP64:
                assert e[k] == eo and np.array_equal(g[k], go)
            else:
                assert abs(e[k] - eo) <= 1e-3 * max(1.0, abs(eo))
                assert np.max(np.abs(g[k] - go)) <= 1e-3 * max(1.0, np.max(np.abs(go)))
    ctx.close()
