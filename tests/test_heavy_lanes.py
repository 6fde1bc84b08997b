"""Models of more than 64 movable atoms, at most 64 of them heavy: the
evaluation's lanes take the heavy atoms alone, so the hydrogens may have no
forces.  Such ligands against the oracle (FP64 bit for bit, FP32 within the
reference's bound for an evaluation away from a discontinuity), and the same
ligands with pairs that hold a hydrogen, which the flattener never makes but
an upload accepts: their lanes take every atom.  A model of hydrogens alone
has nothing but pairs."""
import numpy as np
import pytest

import smina_gpu as sg
from common import eval_confs_mix, gd_c0, heavy_types, oracle_for, receptor

pytestmark = pytest.mark.gpu

V = (10.0, 1000.0, 10.0)


def with_pairs(f, extra):
    """f's flat model with the ligand pairs `extra` after its own"""
    v = sg.FlatModel()
    sg.C.pointer(v)[0] = f.view
    types = np.ctypeslib.as_array(f.view.atom_type, (f.natoms,))
    n = f.npairs
    a, b = (np.ascontiguousarray(np.concatenate([p, [e[k] for e in extra]]), np.int32)
            for k, p in enumerate((f.pair_a, f.pair_b)))
    own = np.ctypeslib.as_array(f.view.pair_tri, (n,)) if n else np.zeros(0, np.int32)
    lo = [min(types[i], types[j]) for i, j in extra]
    hi = [max(types[i], types[j]) for i, j in extra]
    tri = np.ascontiguousarray(np.concatenate([own, [h * (h + 1) // 2 + l for l, h in zip(lo, hi)]]), np.int32)
    v.pair_a, v.pair_b, v.pair_tri = (sg.ptr(x, sg.I32P) for x in (a, b, tri))
    v.npairs = n + len(extra)

    class View:
        pass
    w = View()
    w.view, w.keep = v, (a, b, tri, f)
    return w


def hydrogen_pairs(f):
    """every hydrogen with the others and with the heavy atoms away from it,
    as the pair's first atom and as its second"""
    types = np.ctypeslib.as_array(f.view.atom_type, (f.natoms,))
    h = [int(k) for k in np.where(types <= 1)[0]]
    return [(a, b) for a in range(f.natoms) for b in range(a + 4, f.natoms) if a in h or b in h]


@pytest.fixture(scope="module")
def ctx():
    c = sg.Context(0)
    n, smooth, fast = sg.build_tables(sg.vina_scoring())
    c.upload_tables(n, smooth, fast)
    yield c
    c.close()


def compare(ctx, o, m, bid, f, lig, prec, backend, confs, least=1.0):
    rec, gd = receptor(), gd_c0()
    rid = ctx.upload_receptor(rec.xyz, rec.type)
    kw = dict(receptor_id=rid, gd=gd, slope=10.0) if backend else \
        dict(grid_id=ctx.build_grids(rid, gd, heavy_types(lig), prec))
    n = len(confs)
    e, g, x = ctx.eval_confs(bid, [0] * n, confs, f.change_size, f.natoms, V, **kw)
    for k in range(n):
        eo, go, xo = o.eval_deriv(m, confs[k], V, backend=backend, slope=10.0 if backend else 1e6)
        if prec == sg.FP64:
            assert e[k] == eo and np.array_equal(g[k], go) and np.array_equal(x[k], xo), k
        else:
            assert abs(e[k] - eo) <= 1e-3 * max(least, abs(eo)), k
            assert np.max(np.abs(g[k] - go)) <= 1e-3 * max(least, np.max(np.abs(go))), k


@pytest.mark.parametrize("prec,extra", [(sg.FP64, False), (sg.FP64, True), (sg.FP32, False)],
                         ids=["fp64-own", "fp64-hydrogens", "fp32-own"])
@pytest.mark.parametrize("backend", [0, 1])
@pytest.mark.parametrize("spec", [(3, 63, 12), (9, 64, 12)])
def test_evaluation(ctx, spec, prec, backend, extra):
    lig = sg.Mol.ligand(*spec)
    f = sg.Flat(lig)
    assert f.natoms > 64 and f.nheavy <= 64
    o, ids, _, gd = oracle_for([lig])
    pairs = hydrogen_pairs(f) if extra else []
    for a, b in pairs:
        o.add_ligand_pair(ids[0], a, b)
    bid = ctx.upload_models([with_pairs(f, pairs)], prec)
    confs = eval_confs_mix(f, gd, 16, seed=5)[1::2]
    compare(ctx, o, ids[0], bid, f, lig, prec, backend, confs)


@pytest.mark.parametrize("spec", [(3, 63, 12), (9, 64, 12)])
def test_fp32_forces_on_hydrogens(ctx, spec):
    """what the hydrogens' pairs change, with and without them, so that it
    does not drown in the gradient (the receptor's repulsion capped to 0 for
    the same reason).  The changes are 0.012 to 0.15; the bound 2e-3 is 1e-5 of
    two gradients of up to 50, summed over 70 atoms in FP32, twice over."""
    lig = sg.Mol.ligand(*spec)
    f = sg.Flat(lig)
    rec, v = receptor(), (10.0, 0.0, 10.0)
    pairs = hydrogen_pairs(f)
    o, ids, _, gd = oracle_for([lig, lig])
    for a, b in pairs:
        o.add_ligand_pair(ids[1], a, b)
    rid = ctx.upload_receptor(rec.xyz, rec.type)
    gid = ctx.build_grids(rid, gd, heavy_types(lig), sg.FP32)
    bid = ctx.upload_models([f, with_pairs(f, pairs)], sg.FP32)
    confs = eval_confs_mix(f, gd, 10, seed=5)[1::2]
    n = len(confs)
    e, g, _ = ctx.eval_confs(bid, [0] * n + [1] * n, np.concatenate([confs, confs]), f.change_size, f.natoms, v,
                             grid_id=gid)
    for k in range(n):
        (e0, g0, _), (e1, g1, _) = (o.eval_deriv(i, confs[k], v) for i in ids)
        assert np.max(np.abs(g1 - g0)) > 0.01
        assert np.max(np.abs((g[n + k] - g[k]) - (g1 - g0))) <= 2e-3, k
        assert abs((e[n + k] - e[k]) - (e1 - e0)) <= 2e-3, k


@pytest.mark.parametrize("extra", [False, True], ids=["own", "hydrogens"])
def test_fp64_chain(ctx, extra):
    lig = sg.Mol.ligand(3, 63, 12)
    f = sg.Flat(lig)
    rec, gd = receptor(), gd_c0()
    o, ids, _, _ = oracle_for([lig])
    pairs = hydrogen_pairs(f) if extra else []
    for a, b in pairs:
        o.add_ligand_pair(ids[0], a, b)
    rid = ctx.upload_receptor(rec.xyz, rec.type)
    gid = ctx.build_grids(rid, gd, heavy_types(lig), sg.FP64)
    bid = ctx.upload_models([with_pairs(f, pairs)], sg.FP64)
    c0, s0 = f.make_chain(5, gd)
    cnt, e, c, x, ev = ctx.run_mc(bid, gid, sg.mc_params(), [0], c0[None], s0[None], [3], [12],
                                  coord_stride=3 * f.nheavy)
    eo, co, xo, evo = o.mc_chain(ids[0], sg.mc_params(), 3, 12, c0, s0)
    assert cnt[0] == len(eo) and np.array_equal(e[0, :cnt[0]], eo) and ev[0] == evo


@pytest.mark.parametrize("npairs", [0, 4])
@pytest.mark.parametrize("prec", [sg.FP64, sg.FP32], ids=["fp64", "fp32"])
def test_no_heavy_atoms(ctx, prec, npairs):
    """66 atoms, every one a hydrogen: the energy and gradient of the oracle
    for the same pairs (FP32: relative to them, they are small), zeros
    without any"""
    mol = sg.Mol.ligand(9, 64, 12)
    np.ctypeslib.as_array(mol.desc_ptr.contents.type, (mol.natoms,))[:] = 0
    f = sg.Flat(mol)
    assert f.natoms == 66 and f.nheavy == 0 and f.npairs == 0
    o, ids, _, gd = oracle_for([mol])
    pairs = [(0, 40), (1, 50), (10, 65), (30, 60)][:npairs]
    for a, b in pairs:
        o.add_ligand_pair(ids[0], a, b)
    bid = ctx.upload_models([with_pairs(f, pairs)], prec)
    confs = eval_confs_mix(f, gd, 12, seed=5)
    compare(ctx, o, ids[0], bid, f, sg.Mol.ligand(9, 64, 12), prec, 0, confs, least=0.0)
