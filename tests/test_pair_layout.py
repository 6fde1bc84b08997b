"""The pair-parallel evaluation at the edges of its layout: pair counts of a
whole number of 64-lane chunks and one more or less, neighbour lists padded
to batches of 4 (0 to 3 entries of padding), no pairs at all, and an FP64
model whose pairs don't fit a workgroup's LDS (each atom then evaluates its
pairs itself).  FP64 equals the oracle bit for bit; FP32 is within the
reference's bound for an evaluation away from a discontinuity."""
import numpy as np
import pytest

import smina_gpu as sg
from common import eval_confs_mix, gd_c0, heavy_types, oracle_for, receptor

pytestmark = pytest.mark.gpu


def find_ligand(rem):
    """the first synthetic ligand whose pair count is rem modulo 64"""
    for seed in range(1, 400):
        lig = sg.Mol.ligand(seed, 12 + seed % 16, 2 + seed % 2)
        f = sg.Flat(lig)
        if f.npairs >= 63 and f.npairs % 64 == rem:
            return lig, f
    raise AssertionError("no such ligand")


@pytest.fixture(scope="module")
def ctx():
    c = sg.Context(0)
    n, smooth, fast = sg.build_tables(sg.vina_scoring())
    c.upload_tables(n, smooth, fast)
    yield c
    c.close()


def check(ctx, lig, f, prec, backend, n=8):
    gd, rec = gd_c0(), receptor()
    o, ids, _, _ = oracle_for([lig])
    rid = ctx.upload_receptor(rec.xyz, rec.type)
    kw = dict(receptor_id=rid, gd=gd, slope=10.0) if backend else \
        dict(grid_id=ctx.build_grids(rid, gd, heavy_types(lig), prec))
    bid = ctx.upload_models([f], prec)
    confs = eval_confs_mix(f, gd, n, seed=3)[1::2]  # around the input pose
    n = len(confs)
    e, g, x = ctx.eval_confs(bid, [0] * n, confs, f.change_size, f.natoms, (10.0, 1000.0, 10.0), **kw)
    for k in range(n):
        eo, go, xo = o.eval_deriv(ids[0], confs[k], (10.0, 1000.0, 10.0), backend=backend,
                                  slope=10.0 if backend else 1e6)
        if prec == sg.FP64:
            assert e[k] == eo and np.array_equal(g[k], go) and np.array_equal(x[k], xo)
        else:
            assert abs(e[k] - eo) <= 1e-3 * max(1.0, abs(eo))
            assert np.max(np.abs(g[k] - go)) <= 1e-3 * max(1.0, np.max(np.abs(go)))


@pytest.mark.parametrize("rem", [63, 0, 1])
@pytest.mark.parametrize("prec", [sg.FP64, sg.FP32], ids=["fp64", "fp32"])
def test_pair_counts_around_a_chunk(ctx, rem, prec):
    lig, f = find_ligand(rem)
    check(ctx, lig, f, prec, 0)


@pytest.mark.parametrize("prec", [sg.FP64, sg.FP32], ids=["fp64", "fp32"])
def test_no_pairs(ctx, prec):
    lig = sg.Mol.ligand(5, 8, 0)
    f = sg.Flat(lig)
    assert f.npairs == 0
    check(ctx, lig, f, prec, 0)


@pytest.mark.parametrize("backend", [0, 1])
def test_fp64_pairs_past_lds(ctx, backend):
    lig = sg.Mol.ligand(11, 120, 25)
    f = sg.Flat(lig)
    assert f.npairs > 6000
    check(ctx, lig, f, sg.FP64, backend)
    # the FP32 limit is the smaller one, as it was
    with pytest.raises(sg.SgpuError):
        ctx.upload_models([f], sg.FP32)


def test_fp64_chain_with_pairs_past_lds(ctx):
    lig = sg.Mol.ligand(11, 120, 25)
    f = sg.Flat(lig)
    gd, rec = gd_c0(), receptor()
    o, ids, _, _ = oracle_for([lig])
    rid = ctx.upload_receptor(rec.xyz, rec.type)
    gid = ctx.build_grids(rid, gd, heavy_types(lig), sg.FP64)
    bid = ctx.upload_models([f], sg.FP64)
    c0, s0 = f.make_chain(5, gd)
    cnt, e, c, x, ev = ctx.run_mc(bid, gid, sg.mc_params(), [0], c0[None], s0[None], [2], [8],
                                  coord_stride=3 * f.nheavy)
    eo, co, xo, evo = o.mc_chain(ids[0], sg.mc_params(), 2, 8, c0, s0)
    assert cnt[0] == len(eo) and np.array_equal(e[0, :cnt[0]], eo) and ev[0] == evo


@pytest.mark.parametrize("passes", [1, 2, 3, 4, 5, 6, 7])
@pytest.mark.parametrize("prec", [sg.FP64, sg.FP32], ids=["fp64", "fp32"])
def test_pair_batches(ctx, passes, prec):
    """every mix of whole batches of 4 passes and a shorter last one"""
    for seed in range(1, 400):
        lig = sg.Mol.ligand(seed, 10 + seed % 30, 1 + seed % 5 if seed % 30 > 12 else 1)
        f = sg.Flat(lig)
        if (f.npairs + 63) // 64 == passes:
            return check(ctx, lig, f, prec, 0)
    raise AssertionError("no such ligand")
