"""Leaf emission over its tile sizes (64, 256 or 1024 level-(L-1) nodes per
work-group): against the oracle, bit for bit, at the smallest grids (one part
tile), on ragged DEMs and at the levels where the tile size changes; and the
learned step's unit records with many units, several and one unit per tile."""
import os

import numpy as np
import pytest

import cases
import parity_util

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,xsz,ysz,solver,prec", [
    (2, 4, 3, "mwdg2", "f64"), (3, 8, 8, "hwfv1", "f32"), (4, 13, 16, "mwdg2", "f32"), (5, 32, 27, "hwfv1", "f64"),
    (9, 401, 512, "mwdg2", "f32"), (10, 1024, 700, "hwfv1", "f32"), (10, 600, 1000, "mwdg2", "f64"),
    (11, 1500, 1100, "mwdg2", "f32")])
def test_emission_tiles(case_dir, L, xsz, ysz, solver, prec):
    par = cases.random_case(os.path.join(str(case_dir), f"tile{L}{solver}{prec}"), L=L, seed=7 + L, xsz=xsz, ysz=ysz,
                            solver=solver, manning=0.03, t_end=5.0, wet_frac=0.4,
                            srcs=2 if L > 3 else 0, stage=2 if L > 3 else 0)
    parity_util.run_pair(par, prec, steps=3)


@pytest.mark.parametrize("L", [7, 8, 9, 10, 11])
def test_learned_units_over_tiles(case_dir, L):
    """With every unit frozen the learned step makes the plain step's tree;
    its depths move from it by the rounding of the reconstructions it leaves
    out, some 1e-16 of an elevation of 20 m per step (1e-9 m is far above
    that and far below a wrong maximum, which changes the thresholds)."""
    import mwdg2
    from bench import finest_fields
    par = cases.urban(os.path.join(str(case_dir), f"unit{L}"), L=L, t_end=100.0)
    steps = 24
    with mwdg2.Simulation(par, "f64") as ref:
        ref.step(steps)
        h_ref, leaves_ref = finest_fields(ref, L)[0], ref.get("leaves")
        mx_ref = ref.counters()["maxes"]
    with mwdg2.Mlp(3) as m, mwdg2.Simulation(par, "f64") as s:
        s.set_learned(m, decide_every=8, full_every=32, threshold=2.0)
        s.step(steps)
        h, leaves = finest_fields(s, L)[0], s.get("leaves")
        mx = s.counters()["maxes"]
    assert np.array_equal(leaves, leaves_ref)
    assert float(np.max(np.abs(h - h_ref))) <= 1e-9
    assert np.allclose(mx, mx_ref, rtol=1e-9, atol=0)


@pytest.mark.parametrize("L,solver,prec,limit", [
    (3, "mwdg2", "f64", False), (5, "hwfv1", "f32", False), (8, "mwdg2", "f32", False), (8, "hwfv1", "f64", False),
    (7, "mwdg2", "f64", True), (10, "mwdg2", "f32", True)])
def test_single_stages_make_the_step(case_dir, L, solver, prec, limit):
    """The stages called one by one (encode and decode apart, the limiter's
    largest depth taken from B) give what whole steps give, bit for bit."""
    import mwdg2
    par = cases.random_case(os.path.join(str(case_dir), f"stg{L}{solver}{prec}{limit}"), L=L, seed=3 + L,
                            solver=solver, manning=0.03, t_end=50.0, srcs=3 if L > 3 else 0)
    if limit:
        with open(par, "a") as f:
            f.write("limitslopes\ntol_Krivo     1\n")
    stages = ["prologue", "point_sources", "encode", "decode", "emit", "swap_masks"]
    stages += ["stage1", "encode_scale", "stage2"] if solver == "mwdg2" else ["fv1"]
    with mwdg2.Simulation(par, prec) as a, mwdg2.Simulation(par, prec) as b:
        a.step(3)
        for _ in range(3):
            for name in stages:
                b.stage(name)
        ca, cb = a.counters(), b.counters()
        assert ca["time"] == cb["time"] and ca["dt_next"] == cb["dt_next"] and ca["n_leaves"] == cb["n_leaves"]
        leaves = a.get("leaves")
        assert np.array_equal(leaves, b.get("leaves"))
        assert np.array_equal(a.get("sig")[3:], b.get("sig")[3:])
        for c in ("eta0", "qx0", "qy0") + (("eta1x", "qx1y", "qy1x") if solver == "mwdg2" else ()):
            assert np.array_equal(a.get("A." + c)[leaves], b.get("A." + c)[leaves]), c


@pytest.mark.parametrize("L,eps", [(4, 1e-3), (9, 1e-3), (9, 0.0), (10, 0.0), (11, 1e-4)])
def test_wet_lists_full_and_in_one_part(case_dir, L, eps):
    """Every leaf wet (each region of the wet lists holds all its share), from
    the emission (epsilon > 0) and from the sweeps (epsilon 0); at the largest
    level a small DEM in one corner of the mesh, so that few regions hold it all."""
    side = {11: 200}.get(L)
    par = cases.random_case(os.path.join(str(case_dir), f"full{L}{eps}"), L=L, seed=41 + L, eps=eps, manning=0.03,
                            t_end=50.0, wet_frac=1.0, xsz=side, ysz=side)
    parity_util.run_pair(par, "f32", steps=3)


@pytest.mark.parametrize("L,prec", [(4, "f32"), (4, "f64"), (5, "f32"), (6, "f32"), (6, "f64"), (7, "f32")])
def test_hwfv1_small_trees(case_dir, L, prec):
    """HWFV1's whole tree in one work-group (4 to 6 parent levels) and one level
    above it: the oracle's, bit for bit, on a full grid over enough steps for the
    tree to change; and the stages apart make the same."""
    import mwdg2
    par = cases.random_case(os.path.join(str(case_dir), f"hw{L}{prec}"), L=L, seed=50 + L, solver="hwfv1",
                            manning=0.03, t_end=50.0, wet_frac=0.5, srcs=2, stage=2)
    parity_util.run_pair(par, prec, steps=6)
    with mwdg2.Simulation(par, prec) as a, mwdg2.Simulation(par, prec) as b:
        a.step(4)
        for _ in range(4):
            for name in ["prologue", "point_sources", "encode", "decode", "emit", "swap_masks", "fv1"]:
                b.stage(name)
        ca, cb = a.counters(), b.counters()
        assert ca["time"] == cb["time"] and ca["dt_next"] == cb["dt_next"] and ca["n_leaves"] == cb["n_leaves"]
        leaves = a.get("leaves")
        assert np.array_equal(leaves, b.get("leaves"))
        assert np.array_equal(a.get("sig")[3:], b.get("sig")[3:])
        for c in ("eta0", "qx0", "qy0"):
            assert np.array_equal(a.get("A." + c), b.get("A." + c)), c


@pytest.mark.parametrize("L,prec", [(3, "f64"), (5, "f32"), (6, "f64"), (8, "f32"), (9, "f64"), (10, "f32")])
def test_hwfv1_update_after_whole_steps(case_dir, L, prec):
    """The neighbour lists after whole HWFV1 steps are those of the last step's
    leaves, whichever kernels made it: the update stage called on its own reads
    them and gives what it gives after an emission of its own; new labels (the
    decode called on its own) leave them alone; and uploaded lists stay as they
    were uploaded, one after the other."""
    import mwdg2
    par = cases.random_case(os.path.join(str(case_dir), f"upd{L}{prec}"), L=L, seed=60 + L, solver="hwfv1",
                            manning=0.03, t_end=50.0, wet_frac=0.5, srcs=2 if L > 3 else 0, stage=2 if L > 3 else 0)
    with mwdg2.Simulation(par, prec) as a, mwdg2.Simulation(par, prec) as b, mwdg2.Simulation(par, prec) as c:
        for sim in (a, b, c):
            sim.step(3)
        a.stage("fv1")
        b.stage("emit")
        nbrs = [b.get(f"nbr{k}") for k in range(4)]
        b.stage("fv1")
        ca, cb = a.counters(), b.counters()
        assert ca["time"] == cb["time"] and ca["dt_next"] == cb["dt_next"] and ca["n_leaves"] == cb["n_leaves"]
        for v in ("eta0", "qx0", "qy0"):
            assert np.array_equal(a.get("A." + v), b.get("A." + v)), v
        for name in ("prologue", "encode", "decode"):
            c.stage(name)
        for k in range(4):
            assert np.array_equal(a.get(f"nbr{k}"), nbrs[k])
            assert np.array_equal(c.get(f"nbr{k}"), nbrs[k])
        for k in range(4):
            c.set(f"nbr{k}", nbrs[(k + 1) % 4])
        for k in range(4):
            assert np.array_equal(c.get(f"nbr{k}"), nbrs[(k + 1) % 4])


@pytest.mark.parametrize("side", [None, 200])
def test_learned_reencode_above_and_in_units(case_dir, side):
    """max_ref_lvl 12: the stage-1 re-encode by level-6 units and, where the
    step has leaves at levels <= 5 (a small DEM in the corner of the mesh), of
    the levels above them: every significant parent of the stage-1 state holds
    what the plain step's holds (1e-9: see test_learned_units_over_tiles)."""
    import mwdg2
    L, steps = 12, 12
    d = os.path.join(str(case_dir), f"reenc{side}")
    par = (cases.urban(d, L=L, t_end=100.0) if side is None else
           cases.random_case(d, L=L, seed=71, manning=0.03, t_end=100.0, wet_frac=0.5, xsz=side, ysz=side - 40))
    with mwdg2.Simulation(par, "f64") as ref, mwdg2.Mlp(3) as m, mwdg2.Simulation(par, "f64") as s:
        s.set_learned(m, decide_every=4, full_every=16, threshold=2.0)
        ref.step(steps)
        s.step(steps)
        sig = ref.get("sig")
        assert np.array_equal(sig[3:], s.get("sig")[3:])
        coarse = int(ref.get("leaves").min()) < parity_util.lvl_idx(6)
        assert coarse == (side is not None)
        nodes = np.flatnonzero(sig)
        nodes = nodes[nodes >= (3 if coarse else parity_util.lvl_idx(6))]
        for c in ("eta0", "eta1x", "qx0", "qy1y"):
            a, b = ref.get("B." + c)[nodes], s.get("B." + c)[nodes]
            assert float(np.max(np.abs(a - b))) <= 1e-9, c


@pytest.mark.parametrize("L,xsz,ysz,solver,prec,limit", [
    (11, 1300, 1090, "hwfv1", "f32", False), (11, 1025, 1200, "hwfv1", "f64", False),
    (12, 300, 260, "hwfv1", "f32", False), (11, 1100, 900, "mwdg2", "f32", True),
    (11, 1030, 1100, "mwdg2", "f64", True)])
def test_flat_levels(case_dir, L, xsz, ysz, solver, prec, limit):
    """Levels from 10 on are flat launches in the encode, the decode and the
    stage-1 re-encode: one of them (max_ref_lvl 11) and two (12, with 1024-node
    emission tiles), for HWFV1 and for MWDG2 with the limiter, against the
    oracle bit for bit."""
    par = cases.random_case(os.path.join(str(case_dir), f"flat{L}{solver}{prec}"), L=L, seed=90 + L, xsz=xsz, ysz=ysz,
                            solver=solver, manning=0.03, t_end=20.0, wet_frac=0.4, srcs=2, stage=2)
    if limit:
        with open(par, "a") as f:
            f.write("limitslopes\ntol_Krivo     1\n")
    parity_util.run_pair(par, prec, steps=3)


def _level_of(h):
    return np.floor(np.log2(3 * (h.astype(np.int64) - 3) + 1) / 2).astype(np.int64)


def _part1(v):
    v = v.astype(np.int64)
    for s, m in ((8, 0x00FF00FF), (4, 0x0F0F0F0F), (2, 0x33333333), (1, 0x55555555)):
        v = (v | (v << s)) & m
    return v


def _compact(c):
    c = c.astype(np.int64) & 0x55555555
    for s, m in ((1, 0x33333333), (2, 0x0F0F0F0F), (4, 0x00FF00FF), (8, 0x0000FFFF)):
        c = (c | (c >> s)) & m
    return c


@pytest.mark.parametrize("solver", ["mwdg2", "hwfv1"])
def test_scanned_tile_counts(case_dir, solver):
    """Above 4096 emission tiles (max_ref_lvl 13) their leaf counts are scanned
    by a launch of its own. A long thin DEM across the mesh puts leaves of every
    level into tiles all along the list: the leaf list is the one that the mask
    gives (in Morton order), and the neighbours are those of the finest cells
    beside a leaf, by search in that list."""
    import mwdg2
    L, xsz, ysz = 13, 8000, 20
    d = os.path.join(str(case_dir), f"scan{solver}")
    par = cases.random_case(d, L=6, seed=5, solver=solver, manning=0.03, t_end=50.0)
    with open(par) as f:
        text = f.read()
    with open(par, "w") as f:
        f.write("\n".join(f"max_ref_lvl   {L}" if e.split()[:1] == ["max_ref_lvl"] else e
                          for e in text.splitlines()) + "\n")
    x = np.arange(xsz)[None, :]
    z = (2.0 + np.sin(x / 300.0) + 0.3 * np.sin(x / 7.0) + 0.1 * cases.uniform(6, xsz * ysz).reshape(ysz, xsz))
    cases.write_raster(os.path.join(d, "case.dem"), z, 0.0, 0.0, 1.0)
    cases.write_raster(os.path.join(d, "case.start"), np.maximum(0.0, 2.0 - z), 0.0, 0.0, 1.0)
    start_of = np.array([parity_util.lvl_idx(l) for l in range(L + 1)])
    with mwdg2.Simulation(par, "f32") as s:
        for _ in range(2):
            s.step(2)
            leaves, sig, c = s.get("leaves").astype(np.int64), s.get("sig"), s.counters()
            nodes, expect = np.array([0]), []               # Morton codes of the level's nodes of the tree
            for l in range(L + 1):
                inner = sig[start_of[l] + nodes] != 0 if l < L else np.zeros(nodes.size, dtype=bool)
                expect.append(start_of[l] + nodes[~inner])
                nodes = (4 * nodes[inner][:, None] + np.arange(4)[None, :]).ravel()
            expect = np.concatenate(expect)
            lev = _level_of(expect)
            first = (expect - start_of[lev]) << (2 * (L - lev))
            order = np.argsort(first)
            expect, lev, first = expect[order], lev[order], first[order]
            assert c["n_leaves"] == leaves.size > 10000 and np.array_equal(leaves, expect)
            last = first + (1 << (2 * (L - lev))) - 1
            # tiles (64 x 64 cells) that hold a leaf's start: the strip alone lies in 8000 / 64 = 125
            assert np.unique(first >> 12).size >= 125
            xs, ys, xe, ye = _compact(first), _compact(first >> 1), _compact(last), _compact(last >> 1)
            n = 1 << L
            edge_n, edge_e = (ye == n - 1) | (ye == ysz - 1), (xe == n - 1) | (xe == xsz - 1)
            for k, (xn, yn, border) in enumerate(((xe, ye + 1, edge_n), (xe + 1, ye, edge_e),
                                                  (xs, ys - 1, ys == 0), (xs - 1, ys, xs == 0))):
                m = _part1(np.clip(xn, 0, n - 1)) | (_part1(np.clip(yn, 0, n - 1)) << 1)
                ml = np.minimum(lev, lev[np.searchsorted(first, m, side="right") - 1])
                want = np.where(border, -1, start_of[ml] + (m >> (2 * (L - ml))))
                assert np.array_equal(s.get(f"nbr{k}"), want), k
            assert c["steps"] > 0 and c["nonfinite"] == 0 and 0.0 < c["dt_next"] < 10.0
