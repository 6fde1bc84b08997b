"""A launch with more chains than can all speculate, among them a few that
outlast the rest: those run speculative chains in launches of their own, and
every chain of the batch equals the one of a launch without speculation."""
import numpy as np
import pytest

import smina_gpu as sg
from common import gd_c0, heavy_types, receptor

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [sg.FP32, sg.MIXED, sg.FP64], ids=["fp32", "mixed", "fp64"])
def test_the_longest_chains_speculate(prec, monkeypatch, capfd):
    gd, rec = gd_c0(), receptor()
    ligs = [sg.Mol.ligand(2, 38, 9), sg.Mol.ligand(4, 50, 10)] + [sg.Mol.ligand(10 + k, 10, 2) for k in range(8)]
    flats = [sg.Flat(m) for m in ligs]
    ctx = sg.Context(0)
    n, smooth, fast = sg.build_tables(sg.vina_scoring())
    ctx.upload_tables(n, smooth, fast)
    rid = ctx.upload_receptor(rec.xyz, rec.type)
    gid = ctx.build_grids(rid, gd, heavy_types(*ligs), sg.FP64 if prec == sg.FP64 else sg.FP32)
    bid = ctx.upload_models(flats, prec)
    _, cus = ctx.device_info()
    # 8 chains of each long ligand, the rest small: 14 waves per CU in all,
    # past what could speculate at width 2
    models = [0] * 8 + [1] * 8 + [2 + k % 8 for k in range(14 * cus - 16)]
    cs = max(f.conf_size for f in flats)
    seeds = [flats[m].make_chain(50 + k % 64, gd) for k, m in enumerate(models)]
    confs = np.zeros((len(models), cs))
    for k, (c, _) in enumerate(seeds):
        confs[k, :len(c)] = c
    rngs = np.array([s for _, s in seeds])
    steps = [12 if m < 2 else 1 for m in models]
    iters = [(25 + flats[m].natoms) // 3 for m in models]
    monkeypatch.setenv("SGPU_LOG_PLAN", "1")
    out = {}
    for spec in (None, "1"):
        if spec:
            monkeypatch.setenv("SGPU_SPEC", spec)
        out[spec] = ctx.run_mc(bid, gid, sg.mc_params(), models, confs, rngs, steps, iters,
                               coord_stride=3 * max(f.nheavy for f in flats))
        log = capfd.readouterr().err
        assert ("one speculative chain" in log) == (spec is None), log
        assert "chains" in log or "workgroup," in log
    for a, b in zip(out[None], out["1"]):
        assert np.array_equal(a, b)
    ctx.close()
