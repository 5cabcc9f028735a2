"""Which form of the step kernels runs: on either side of the sizes up to which
plans and pools take the block form by themselves, what a pool says of its next
launch before any has run, and what the tuner makes of it."""

from __future__ import annotations

import numpy as np
import pytest

import fdtd2d_amd as F
from fdtd2d_amd import batch
from fdtd2d_amd.tuning import ShapeCache, mix_key

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
