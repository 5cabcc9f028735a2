"""Reads and writes of fields whose rows are not contiguous on the device, next
to work queued elsewhere on it: they wait for the launches their own shot or
plan depends on and for no others."""

from __future__ import annotations

import numpy as np
import pytest

import fdtd2d_amd as F
from oracle.oracle import Oracle

from helpers import random_problem

pytestmark = pytest.mark.gpu

FIELDS = (F.EZ, F.HX, F.HY, F.JZ)


def _bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


def _add_long(pool):
    """A 4000^2 shot: its 5000 launches take about 0.6 s on the device and a
    tenth of that to issue."""
    return pool.add(F.Setup.box(4000, 4000, 12, 40000, 1e-3))


def test_finished_shot_is_read_while_others_run(gpu_device):
    """Every field of a finished shot of odd width, while the last launches of
    another shot of the pool are still queued."""
    p = random_problem(np.random.default_rng(41), nx=301, ny=203, npml=8, nsteps=8, table=False)
    ref = Oracle(p, 32)
    ref.run(p.nsteps)
    with F.Pool(gpu_device) as pool:
        big = _add_long(pool)
        sid = pool.add(p)
        pool.step(8)
        pool.sync()
        pool.step(5000)
        got = [pool.read_field(sid, w) for w in FIELDS]
        done = pool.state(big)
        print(f"4000^2 shot beside it: {done}", flush=True)
        assert done[0] == done[1] and not done[2]  # all issued, not yet complete
    for w, g in zip(FIELDS, got):
        assert np.array_equal(_bits(g), _bits(ref.read_field(w))), w


def test_plan_is_read_and_written_while_a_pool_runs(gpu_device):
    """Fields and psi strips of a plan of odd width, read and written beside a
    pool's queued launches."""
    p = random_problem(np.random.default_rng(42), nx=301, ny=203, npml=8, nsteps=8, table=False)
    ref = Oracle(p, 32)
    ref.run(p.nsteps)
    with F.Plan(p, gpu_device) as plan, F.Pool(gpu_device) as pool:
        plan.run(p.nsteps)
        plan.sync()
        big = _add_long(pool)
        pool.step(8)
        pool.sync()
        pool.step(5000)
        got = {w: plan.read_field(w) for w in FIELDS}
        psi = {w: plan.read_psi(w) for w in (F.PSI_HYX, F.PSI_EZX, F.PSI_HXY, F.PSI_EZY)}
        plan.write_field(F.EZ, got[F.EZ])
        plan.write_psi(F.PSI_EZX, psi[F.PSI_EZX])
        done = pool.state(big)
        print(f"4000^2 shot beside it: {done}", flush=True)
        assert done[0] == done[1] and not done[2]
    for w, g in got.items():
        assert np.array_equal(_bits(g), _bits(ref.read_field(w))), w
    for w, g in psi.items():
        assert np.array_equal(_bits(g), _bits(ref.read_psi(w))), w


@pytest.mark.parametrize("nx,ny", [(2049, 2101), (4097, 1100)])
def test_rows_beyond_the_packing_buffer(gpu_device, nx, ny):
    """Planes larger than the 16 MiB packing buffer go through it in parts:
    the last one shorter, Hx and Hy with their shorter sides."""
    assert nx * ny * 4 > 16 << 20
    rng = np.random.default_rng(nx)
    p = F.Setup.box(nx, ny, 6, 4, 1e-3)
    with F.Plan(p, gpu_device) as plan:
        for which in (F.EZ, F.HX, F.HY):
            v = rng.standard_normal(plan.read_field(which).shape).astype(np.float32)
            plan.write_field(which, v)
            assert np.array_equal(_bits(plan.read_field(which)), _bits(v)), which


def test_pool_buffer_grows_with_the_shots_read(gpu_device):
    """Shots of 0.03, 0.24, 2.4 and 17 MB a field (the packing buffer's least
    and most size between them), read in that order and back."""
    rng = np.random.default_rng(43)
    probs = [random_problem(rng, nx=nx, ny=ny, npml=5, nsteps=8, table=False)
             for nx, ny in ((90, 70), (301, 203), (777, 803), (2049, 2101))]
    want = []
    for p in probs:
        ref = Oracle(p, 32, threads=8)
        ref.run(p.nsteps)
        want.append({w: ref.read_field(w) for w in FIELDS})
    with F.Pool(gpu_device) as pool:
        ids = [pool.add(p) for p in probs]
        pool.step(1)
        for k in (0, 1, 2, 3, 2, 1, 0):
            for w in FIELDS:
                assert np.array_equal(_bits(pool.read_field(ids[k], w)), _bits(want[k][w])), (k, w)
