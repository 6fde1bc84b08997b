"""The host side of a docking in batches: ligands and chains past the sizes at
which the host works on several threads give what they give alone (flattening,
chain start states, merging and mode selection), and the packed download
returns every chain's own number of minima."""
import numpy as np
import pytest

import smina_gpu as sg
from common import gd_c0, heavy_types, receptor

pytestmark = pytest.mark.gpu


def test_a_batch_equals_its_ligands_alone():
    rec, gd = receptor(), gd_c0()
    ligs = [sg.Mol.ligand(100 + k, 8 + k % 9, 1 + k % 2) for k in range(70)]
    d = sg.Docking(rec, gd, exhaustiveness=4, seed=3, step_fraction=1.0 / 2048)
    d.prepare(ligs)
    batch = d.dock(ligs, top_coords=True, confs=True)
    for k in (0, 1, 33, 68, 69):
        alone = d.dock([ligs[k]], top_coords=True, confs=True)[0]
        assert alone["e"] == batch[k]["e"] and alone["evals"] == batch[k]["evals"]
        assert np.array_equal(alone["confs"], batch[k]["confs"])
        assert np.array_equal(alone["coords"], batch[k]["coords"])


@pytest.mark.parametrize("saved", [1, 20, 64])
def test_packed_results(saved):
    gd, rec = gd_c0(), receptor()
    ligs = [sg.Mol.ligand(1, 10, 2), sg.Mol.ligand(2, 38, 9)]
    flats = [sg.Flat(m) for m in ligs]
    ctx = sg.Context(0)
    n, smooth, fast = sg.build_tables(sg.vina_scoring())
    ctx.upload_tables(n, smooth, fast)
    rid = ctx.upload_receptor(rec.xyz, rec.type)
    gid = ctx.build_grids(rid, gd, heavy_types(*ligs), sg.FP32)
    bid = ctx.upload_models(flats, sg.FP32)
    cs = max(f.conf_size for f in flats)
    xs = 3 * max(f.nheavy for f in flats)
    steps = [0, 1, 40, 3, 0]  # chains without minima among the others
    models = [0, 1, 0, 1, 1]
    seeds = [flats[m].make_chain(9 + k, gd) for k, m in enumerate(models)]
    confs = np.zeros((5, cs))
    for k, (c, _) in enumerate(seeds):
        confs[k, :len(c)] = c
    rngs = np.array([s for _, s in seeds])

    def run(which):
        return ctx.run_mc(bid, gid, sg.mc_params(num_saved=saved), [models[k] for k in which], confs[which],
                          rngs[which], [steps[k] for k in which], [12] * len(which), max_poses=64, coord_stride=xs)
    cnt, e, c, x, ev = run(list(range(5)))
    assert cnt[0] == 0 and cnt[4] == 0 and 1 <= cnt[2] <= saved
    for k in (1, 2, 3):
        c1, e1, k1, x1, v1 = run([k])
        assert c1[0] == cnt[k] and v1[0] == ev[k]
        assert np.array_equal(e1[0], e[k]) and np.array_equal(k1[0], c[k]) and np.array_equal(x1[0], x[k])
        assert np.all(np.diff(e[k, :cnt[k]]) >= 0)
    ctx.close()
