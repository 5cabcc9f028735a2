"""Which form of the step kernels runs: on either side of the sizes up to which
plans and pools take the block form by themselves, what a pool says of its next
launch before any has run, and what the tuner makes of it."""

from __future__ import annotations

import numpy as np
import pytest

import fdtd2d_amd as F
from fdtd2d_amd import batch
from fdtd2d_amd.tuning import ShapeCache, mix_key
from oracle.oracle import Oracle

from helpers import all_state, random_problem

pytestmark = pytest.mark.gpu


def _problem(nx, ny, table, nsteps=400):
    """An empty grid of either medium."""
    p = F.Setup.box(nx, ny, 4, nsteps, 1e-3).problem()
    if table:
        p.medium_kind = F.MEDIUM_TABLE
        p.material = np.zeros((ny, nx), np.int32)
        p.ca, p.cb, p.ne = (np.array([v], np.float32) for v in (1.0, p.cb0, 0.0))
        p.pec_material, p.density = -1, None
    else:
        p.medium_kind = F.MEDIUM_DENSITY
        p.density = np.zeros((ny, nx), np.float32)
    return p


def test_pool_form_before_any_launch(gpu_device):
    """Two density shots of 7400^2 (109.5 million cells) and of 7450^2 (111),
    two table shots of 6700^2 (89.8) and 6720^2 (90.3): the form the next
    launch takes is known before it, and after shots have joined."""
    for n, table, block in ((7400, False, 1), (7450, False, 0), (6700, True, 1), (6720, True, 0)):
        p = _problem(n, n, table)
        with F.Pool(gpu_device) as pool:
            pool.add(p)
            pool.add(p)
            before = pool.info("block")
            pool.step(1)
            pool.sync()
            print(f"2 x {n}^2 table={table}: {before:.0f}, after a launch {pool.info('block'):.0f}", flush=True)
            assert before == block and pool.info("block") == block
            if block:  # one more passes the limit
                pool.add(_problem(1000, 1000, table))
                assert pool.info("block") == 0


def test_pool_form_while_slicing(gpu_device):
    with F.Pool(gpu_device, slice_cells=150 * 150, slice_every=4) as pool:
        assert pool.info("block") == 0
        pool.add(_problem(200, 200, False))
        pool.add(_problem(100, 100, False))
        assert pool.info("block") == 0
        pool.step(1)
        assert pool.info("block") == 0
        pool.set_option("slice_cells", 0)
        assert pool.info("block") == 1


@pytest.mark.parametrize("n,shots,opts,block", [(7450, 2, {}, False), (300, 3, {"slice_cells": 1e4, "slice_every": 2}, False),
                                                (300, 3, {}, True)])
def test_autotune_tries_the_block_form_only_where_it_runs(gpu_device, n, shots, opts, block):
    """The tuner's block trial is one of launches in that form: pools whose
    launches stream by the rule (too many cells, time slicing) have none."""
    p = _problem(n, n, False)
    with F.Pool(gpu_device, **opts) as pool:
        for _ in range(shots):
            pool.add(p)
        rec = batch.autotune(pool, launches_per_trial=1, axes=[("tblock", [8]), ("band", [256, 128])])
        assert any("block" in shape for shape, _ in rec["trials"]) == block
        assert rec["rate"] > 0
        assert pool.info("block") == (1 if "block" in rec["shape"] else 0)


def test_run_pool_of_few_shots_keeps_the_block_form(gpu_device, tmp_path):
    """Five shots whose size shares are those of a shipped streaming shape,
    tuned on 344 million cells: that shape is not theirs."""
    shots = [F.Setup.box(n, n, 4, 240, 1e-3) for n in (1024, 2000, 2000, 2000, 2000)]
    cache = ShapeCache(tmp_path / "shapes.json")
    key = mix_key(batch.shot_sizes(shots))
    assert cache.lookup("pool", key, 256, nearest=True)[0] is not None
    pool, ids, st = batch.run_pool(shots, gpu_device, cache=cache)
    with pool:
        print(st["tuned"]["key"], st["tuned"]["shape"], flush=True)
        assert st["tuned"]["source"] == "trials" and st["tuned"]["shape"].get("block") == 1
        assert all(pool.state(i)[2] for i in ids)
    pool, ids, st = batch.run_pool(shots, gpu_device, cache=cache)
    with pool:
        assert st["tuned"]["trials"] == [] and st["tuned"]["shape"].get("block") == 1


@pytest.mark.parametrize("table,below,above", [(False, 3872, 3874), (True, 4898, 4900)])
def test_plan_limits(gpu_device, table, below, above):
    """Grids just below and above 15 million cells (density), 24 million (table)."""
    for n, block in ((below, 1), (above, 0)):
        with F.Plan(_problem(n, n, table, nsteps=8), gpu_device) as plan:
            assert plan.info("block") == block
            plan.run(8)
            plan.sync()


def _same(got, want, label):
    """Equal bits, where neither is a NaN; those in the same places."""
    for k in want:
        g, w = (np.asarray(v, np.float32) for v in (got[k], want[k]))
        assert np.array_equal(np.isnan(g), np.isnan(w)), f"{label}: {k}: NaN elsewhere"
        ok = ~np.isnan(w)
        assert np.array_equal(g[ok].view(np.uint32), w[ok].view(np.uint32)), f"{label}: {k} differs"


@pytest.mark.parametrize("table", [False, True])
def test_infinities_and_nan_cross_tile_edges(gpu_device, table):
    """Infinities, a NaN and the largest values put beside the edges of tiles
    and of their waves' rows, in plasma and out of it: they spread one cell a
    step and no further, in every shape of either form."""
    p = random_problem(np.random.default_rng(31 + table), nx=420, ny=230, npml=8, nsteps=21, table=table)
    ez = np.zeros((p.ny, p.nx), np.float32)
    # a first column piece ends at 56; a further one stores 48, 112 columns wide
    # ones follow; rows of a wave end every 2, 3, 4 or 6, those of a tile at 16 .. 64
    for j, i, v in ((39, 55, np.inf), (40, 168, -np.inf), (103, 104, np.nan), (119, 56, 3e38), (64, 167, -3e38),
                    (160, 279, np.inf), (199, 391, np.nan)):
        ez[j, i] = v
    ref = Oracle(p, 32, threads=4)
    ref.write_field(F.EZ, ez)
    ref.run(p.nsteps)
    want = all_state(ref, p.npml)
    wild = ~np.isfinite(want["ez"])
    assert 1000 < wild.sum() < 0.5 * wild.size
    for shape in (0, 3, 4) if table else (0, 2, 3, 4):
        with F.Plan(p, gpu_device) as plan:
            plan.set_option("block", shape)
            assert plan.info("block") == (shape > 0)
            plan.write_field(F.EZ, ez)
            for n in (8, 5, 8):
                plan.run(n)
            _same(all_state(plan, p.npml), want, f"shape {shape}")


def test_block_form_with_slicing(gpu_device):
    """The block form switched on in a time-sliced pool: the two alternating
    shot sets, tails at turns, slicing switched off on the way."""
    rng = np.random.default_rng(61)
    sizes = [(100, 90), (310, 320), (140, 77), (301, 330), (90, 130)]
    probs = [random_problem(rng, nx=nx, ny=ny, npml=int(rng.choice([0, 5, 12])), nsteps=int(rng.integers(40, 75)),
                            table=False) for nx, ny in sizes]
    with F.Pool(gpu_device, graph_chunk=4, slice_cells=250 * 250, slice_every=3) as pool:
        ids = [pool.add(p) for p in probs[:4]]
        assert pool.info("block") == 0
        pool.set_option("block", 1)
        assert pool.info("block") == 1
        pool.step(5)
        assert pool.info("block") == 1 and pool.info("list_switches") > 0
        ids.append(pool.add(probs[4]))
        pool.step(6)
        pool.set_option("slice_cells", 0)
        while pool.info("running") > 0:
            pool.step(4)
        pool.sync()
        for sid, p in zip(ids, probs):
            ref = Oracle(p, 32, threads=4)
            ref.run(p.nsteps)
            det, comp = pool.read_detectors(sid)
            rdet, rcomp = ref.read_detectors()
            got = {"det": det, "comp": comp, **{w: pool.read_field(sid, w) for w in (F.EZ, F.HX, F.HY, F.JZ)}}
            want = {"det": rdet, "comp": rcomp, **{w: ref.read_field(w) for w in (F.EZ, F.HX, F.HY, F.JZ)}}
            _same(got, want, f"shot {sid} {p.nx}x{p.ny} steps {p.nsteps}")
