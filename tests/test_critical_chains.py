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


def test_tuner_keeps_only_plans_that_ran(monkeypatch, capfd):
    """A request of four size classes whose longest chains speculate in
    launches of their own: the smallest classes join the next one's launch,
    and the report shows them by that launch's plan; their candidate's plan,
    which never ran, is not kept.  A small request, whose every chain
    speculates, keeps none either."""
    gd, rec = gd_c0(), receptor()
    shapes = [(10, 2)] * 6 + [(38, 9), (48, 9), (60, 14), (80, 18), (50, 10)]
    ligs = [sg.Mol.ligand(30 + k, *s) for k, s in enumerate(shapes)]
    flats = [sg.Flat(m) for m in ligs]
    size_class = [sum(f.npairs > b for b in (256, 512, 1024)) for f in flats]
    assert size_class == [0] * 6 + [1, 2, 3, 3, 2]
    n, smooth, fast = sg.build_tables(sg.vina_scoring())
    cs, xs = max(f.conf_size for f in flats), 3 * max(f.nheavy for f in flats)
    monkeypatch.setenv("SGPU_LOG_PLAN", "1")

    def context():
        ctx = sg.Context(0)
        ctx.upload_tables(n, smooth, fast)
        rid = ctx.upload_receptor(rec.xyz, rec.type)
        return ctx, ctx.build_grids(rid, gd, heavy_types(*ligs), sg.FP32), ctx.upload_models(flats, sg.FP32)

    def request(models):
        seeds = [flats[m].make_chain(50 + k % 64, gd) for k, m in enumerate(models)]
        confs = np.zeros((len(models), cs))
        for k, (c, _) in enumerate(seeds):
            confs[k, :len(c)] = c
        # two ligands of many iterations, among them one of class 3 and one of class 2
        return models, confs, np.array([s for _, s in seeds]), [{9: 24, 10: 30}.get(m, 4) for m in models]

    def plans(text):
        return [(int(k), int(w), s != "") for k, w, s in re.findall(
            r"mc class (\d+): \d+ models, (\d+) waves/workgroup( \(one speculative chain\))?,", text)]

    def launches(ctx, gid, bid, models):
        capfd.readouterr()
        m, confs, rngs, iters = request(models)
        ctx.run_mc(bid, gid, sg.mc_params(), m, confs, rngs, [2] * len(m), iters, coord_stride=xs)
        return plans(capfd.readouterr().err)

    ctx, gid, bid = context()
    _, cus = ctx.device_info()
    many = [9] * 8 + [10] * 8 + [m for m in (6, 7, 8) for _ in range(16)] + [k % 6 for k in range(14 * cus - 64)]
    default = launches(ctx, gid, bid, many)
    m, confs, rngs, iters = request(many)
    rep = ctx.tune_mc(bid, gid, sg.mc_params(), m, confs, rngs, iters, probe_steps=2)
    probes = plans(capfd.readouterr().err)
    ran = {k for k, _, s in probes if not s}
    print(default, sorted(set(probes)), rep, flush=True)
    assert any(s for _, _, s in default) and len(default) <= 4
    joined = [c for c in rep if c["class"] not in ran]
    assert [c["class"] for c in rep] == [0, 1, 2, 3] and joined and 3 in ran
    for c in joined:
        into = next(d for d in rep if d["class"] > c["class"] and d["class"] in ran)
        assert c["candidates"] == into["candidates"] and c["chosen"] == into["chosen"]
    # a request of the smallest ligands alone runs by its default, as before
    few = [k % 6 for k in range(14 * cus)]
    tuned = launches(ctx, gid, bid, few)
    ctx.close()
    ctx, gid, bid = context()
    assert launches(ctx, gid, bid, few) == tuned
    ctx.close()
    ctx, gid, bid = context()
    m, confs, rngs, iters = request([0, 1, 6, 7])
    for c in ctx.tune_mc(bid, gid, sg.mc_params(), m, confs, rngs, iters, probe_steps=2):
        assert all((x["waves"], x["persistent"]) == (1, False) for x in c["candidates"])
    assert launches(ctx, gid, bid, many) == default
    ctx.close()


def test_the_default_workgroups_are_near_the_best():
    """64 ligands of 10-60 heavy atoms x 32 chains in mixed precision: the
    default plan's probe takes no more than 1.15 times the best candidate's
    (1.3 times with the largest workgroup among the most resident)"""
    rng = np.random.default_rng(74)
    heavy = rng.integers(10, 61, 64)
    ligs = [sg.Mol.ligand(100 + k, int(h), int(min(5, (h - 2) // 4))) for k, h in enumerate(heavy)]
    d = sg.Docking(receptor(), sg.grid_dims((0.0, 0.0, 0.0), (26.0, 26.0, 26.0)), precision=sg.MIXED, exhaustiveness=32,
                   seed=1, step_fraction=1.0 / 512)
    d.prepare(ligs)
    ms = [c["ms"] for c in d.tune(ligs, probe_steps=64)[0]["candidates"]]
    print(ms, flush=True)
    assert ms[0] <= 1.15 * min(ms), ms


def test_workgroups_of_a_class_that_lds_bounds(monkeypatch, capfd):
    """a ligand of 66 heavy atoms, whose single chains hold fewer of a CU than
    workgroups do: alone it takes the largest workgroup of the most resident,
    among other ligands of more work the smallest that keeps them; a request
    that does not fill the device takes the largest, too"""
    ligs = [sg.Mol.ligand(67, 66, 14), sg.Mol.ligand(30, 10, 2)]
    monkeypatch.setenv("SGPU_SPEC", "1")
    waves = []
    for models in ([0] * 2304, [0] * 768 + [1] * 4608, [0] * 512):
        flats = [sg.Flat(m) for m in ligs]
        ctx = sg.Context(0)
        n, smooth, fast = sg.build_tables(sg.vina_scoring())
        ctx.upload_tables(n, smooth, fast)
        rid = ctx.upload_receptor(receptor().xyz, receptor().type)
        gd = gd_c0()
        gid = ctx.build_grids(rid, gd, heavy_types(*ligs), sg.FP32)
        bid = ctx.upload_models(flats, sg.FP32)
        seeds = [[f.make_chain(50 + k, gd) for k in range(8)] for f in flats]
        confs = np.zeros((len(models), max(f.conf_size for f in flats)))
        for k, m in enumerate(models):
            confs[k, :flats[m].conf_size] = seeds[m][k % 8][0]
        monkeypatch.setenv("SGPU_LOG_PLAN", "1")
        ctx.run_mc(bid, gid, sg.mc_params(), models, confs, np.array([seeds[m][k % 8][1] for k, m in enumerate(models)]),
                   [1] * len(models), [5] * len(models), coord_stride=3 * max(f.nheavy for f in flats))
        ctx.close()
        waves.append(int(re.search(r"mc class 3: \d+ models, (\d+) waves/workgroup,", capfd.readouterr().err).group(1)))
    print(waves, flush=True)
    assert waves[0] > waves[1] and waves[2] == 2, waves
