"""A launch with more chains than can all speculate, among them a few that
outlast the rest: those run speculative chains in launches of their own, and
every chain of the batch equals the one of a launch without speculation."""
import re

import numpy as np
import pytest

import smina_gpu as sg
from common import gd_c0, heavy_types, receptor

pytestmark = pytest.mark.gpu


def launch(prec, ligs, models, steps, monkeypatch, capfd):
    """the chains with and without speculation: both results, and the plan of
    the first as (group, models, waves, speculative) of each launch"""
    gd, rec = gd_c0(), receptor()
    flats = [sg.Flat(m) for m in ligs]
    ctx = sg.Context(0)
    n, smooth, fast = sg.build_tables(sg.vina_scoring())
    ctx.upload_tables(n, smooth, fast)
    rid = ctx.upload_receptor(rec.xyz, rec.type)
    gid = ctx.build_grids(rid, gd, heavy_types(*ligs), sg.FP64 if prec == sg.FP64 else sg.FP32)
    bid = ctx.upload_models(flats, prec)
    cs = max(f.conf_size for f in flats)
    seeds = [flats[m].make_chain(50 + k % 64, gd) for k, m in enumerate(models)]
    confs = np.zeros((len(models), cs))
    for k, (c, _) in enumerate(seeds):
        confs[k, :len(c)] = c
    rngs = np.array([s for _, s in seeds])
    iters = [(25 + flats[m].natoms) // 3 for m in models]
    monkeypatch.setenv("SGPU_LOG_PLAN", "1")
    out, plans = [], []
    for spec in (None, "1"):
        if spec:
            monkeypatch.setenv("SGPU_SPEC", spec)
        out.append(ctx.run_mc(bid, gid, sg.mc_params(), models, confs, rngs, steps, iters,
                              coord_stride=3 * max(f.nheavy for f in flats)))
        plans.append([(int(k), int(m), int(w), s != "") for k, m, w, s in re.findall(
            r"mc class (\d+): (\d+) models, (\d+) waves/workgroup( \(one speculative chain\))?,",
            capfd.readouterr().err)])
    ctx.close()
    assert not any(s for _, _, _, s in plans[1])
    assert sum(m for _, m, _, _ in plans[1]) == len(set(models))
    return out, plans[0]


@pytest.mark.parametrize("prec", [sg.FP32, sg.MIXED, sg.FP64], ids=["fp32", "mixed", "fp64"])
def test_the_longest_chains_speculate(prec, monkeypatch, capfd):
    ligs = [sg.Mol.ligand(2, 38, 9), sg.Mol.ligand(4, 50, 10)] + [sg.Mol.ligand(10 + k, 10, 2) for k in range(8)]
    ctx = sg.Context(0)
    _, cus = ctx.device_info()
    ctx.close()
    # 8 chains of each long ligand, the rest small: 14 waves per CU in all,
    # past what could speculate at width 2
    models = [0] * 8 + [1] * 8 + [2 + k % 8 for k in range(14 * cus - 16)]
    (a, b), plan = launch(prec, ligs, models, [12 if m < 2 else 1 for m in models], monkeypatch, capfd)
    # launches of their own for both long ligands, at widths 2 or 4; the
    # small ones run alone
    assert sum(m for _, m, w, s in plan if s and w in (2, 4)) >= 2, plan
    assert any(not s for _, _, _, s in plan), plan
    for x, y in zip(a, b):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("largest,second", [((106, 22), (90, 20)), ((106, 22), (104, 18)), ((108, 22), (100, 20))])
def test_a_very_large_fp64_ligand_beside_smaller_ones(largest, second, monkeypatch, capfd):
    """A ligand whose FP64 pairs don't fit LDS beside one whose pairs do: a
    group of speculative chains has a plan of its own, with its pairs in LDS
    where the whole batch's are not, and its workgroups must fit all the
    same (90 heavy atoms at width 2 with their pairs: about 200 KB)."""
    ligs = [sg.Mol.ligand(105, *largest), sg.Mol.ligand(91, *second)] + \
        [sg.Mol.ligand(200 + k, 20, 4) for k in range(60)]
    models = [m for m in range(len(ligs)) for _ in range(8)]
    flats = [sg.Flat(m) for m in ligs[:3]]
    full = [sg.search_params(f.natoms, f.ntors_total)[0] for f in flats]
    steps = [max(1, round(8 * full[min(m, 2)] / full[0])) for m in models]
    (a, b), plan = launch(sg.FP64, ligs, models, steps, monkeypatch, capfd)
    assert any(s for _, _, _, s in plan), plan
    for x, y in zip(a, b):
        assert np.array_equal(x, y)
