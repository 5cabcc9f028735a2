"""The block form of the step kernels (a tile in registers for a whole launch)
against the FP32 oracle, bit for bit, at the sizes where a tile, a wave's rows
or the recomputed columns end: windows of 64 and 128 columns, 24, 32, 36 and 64
rows, grids one cell around them, events in every corner of a tile, RC probes
and the processing line inside interior tiles, partial launches."""

from __future__ import annotations

import numpy as np
import pytest

import fdtd2d_amd as F
from oracle.oracle import Oracle

from helpers import all_state, random_problem
from test_zz_no_alloc import _DeviceBuffer

pytestmark = pytest.mark.gpu

# "block" option: the compiled shapes of each medium
SHAPES = {False: [2, 3, 4], True: [3, 4]}


def _bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


def _check(p, shapes, launches, label, gpu_device):
    ref = Oracle(p, 32, threads=4)
    ref.run(p.nsteps)
    want = all_state(ref, p.npml)
    extra = {}
    if p.rc_i.size:
        extra["rc"] = np.asarray(ref.read_rc())
    if p.line_size:
        extra["line"] = np.asarray(ref.read_line())
    for shape in shapes:
        with F.Plan(p, gpu_device) as plan:
            plan.set_option("block", shape)
            assert plan.info("block") == 1
            for n in launches:
                plan.run(n)
            plan.run(p.nsteps - sum(launches))
            got = all_state(plan, p.npml)
            for k in want:
                assert np.array_equal(_bits(want[k]), _bits(got[k])), f"{label} shape {shape}: {k} differs"
            if "rc" in extra:
                assert np.array_equal(plan.read_rc(), extra["rc"]), f"{label} shape {shape}: rc differs"
            if "line" in extra:
                assert np.array_equal(_bits(plan.read_line()), _bits(extra["line"])), f"{label} shape {shape}: line"


@pytest.mark.parametrize("table", [False, True])
@pytest.mark.parametrize("nx,ny,npml", [(24, 24, 0), (63, 25, 5), (64, 24, 2), (65, 37, 0), (112, 33, 8), (121, 63, 8),
                                        (128, 64, 11), (177, 65, 5), (240, 101, 12), (333, 131, 3)])
def test_edges(gpu_device, nx, ny, npml, table):
    rng = np.random.default_rng(nx * 1000 + ny + table)
    p = random_problem(rng, nx=nx, ny=ny, npml=npml, nsteps=21, table=table)
    _check(p, SHAPES[table], [8, 1], f"{nx}x{ny} P={npml}", gpu_device)


@pytest.mark.parametrize("seed", range(3))
def test_events_captures_and_odd_den(gpu_device, seed):
    """Sources that share a cell, detectors on every row of a wave, RC probes
    and the processing line in interior tiles, den that differs inside."""
    rng = np.random.default_rng(7100 + seed)
    p = random_problem(rng, nx=420, ny=300, npml=8, nsteps=27, table=bool(seed & 1), nsrc=6, ndet=40, ncomp=8)
    p.src_table = p.src_table * 50
    p.src_i[1], p.src_j[1] = p.src_i[0], p.src_j[0]
    p.det_i[:20], p.det_j[:20] = 200, 140 + np.arange(20)
    p.comp_i[0], p.comp_j[0] = p.src_i[0] % 419, p.src_j[0] % 299
    p.rc_imax = np.array([60, 128, 240, 300], np.int32)
    p.rc_i = p.rc_imax + np.arange(4, dtype=np.int32)
    p.rc_jcut, p.rc_level, p.rc_edge0 = 60, 0.07, 1e-3
    p.line_size, p.line_i0, p.line_j, p.line_begin, p.line_end = 180, 100, 150, 3, 25
    if seed == 2:
        p.den_ex, p.den_hy = p.den_ex.copy(), p.den_hy.copy()
        p.den_ex[230] *= np.float32(1.25)
        p.den_hy[190:193] *= np.float32(0.8)
    _check(p, SHAPES[bool(seed & 1)], [5, 8], f"seed {seed}", gpu_device)


def test_more_events_than_lanes_keeps_the_streaming_form(gpu_device):
    """A wave with more than 64 events in its rows: the plan stays with the
    streaming form and still matches."""
    rng = np.random.default_rng(5)
    p = random_problem(rng, nx=150, ny=120, npml=6, nsteps=18, table=False, ndet=70)
    p.det_i[:], p.det_j[:] = 20 + np.arange(70) % 30, 60  # all in the first tile (columns 0..63)
    ref = Oracle(p, 32)
    ref.run(p.nsteps)
    want = all_state(ref, p.npml)
    with F.Plan(p, gpu_device) as plan:
        assert plan.info("block") == 0
        plan.run(p.nsteps)
        got = all_state(plan, p.npml)
    for k in want:
        assert np.array_equal(_bits(want[k]), _bits(got[k])), k


def test_default_form_and_options(gpu_device):
    """Small grids take the block form; an option of the streaming form, or
    block = 0, leaves it; both forms can follow each other in one run."""
    rng = np.random.default_rng(6)
    p = random_problem(rng, nx=200, ny=180, npml=6, nsteps=40, table=False)
    ref = Oracle(p, 32)
    ref.run(p.nsteps)
    want = all_state(ref, p.npml)
    with F.Plan(p, gpu_device) as plan:
        assert plan.info("block") == 1
        plan.run(11)
        plan.set_option("cols_per_lane", 2)
        assert plan.info("block") == 0
        plan.run(13)
        plan.set_option("block", 1)
        assert plan.info("block") == 1
        plan.run(16)
        got = all_state(plan, p.npml)
        with pytest.raises(F.FDTD2DError):
            plan.set_option("block", 9)
    for k in want:
        assert np.array_equal(_bits(want[k]), _bits(got[k])), k


def test_static_lists_limit(gpu_device):
    """A plan in the caller's memory on a long narrow grid, whose smallest
    block tiles (about 23000 of 48 bytes) exceed the 1 MiB static list array,
    keeps the streaming form; a small grid's run from that array."""
    for nx, ny, block in ((130, 250000, 0), (200, 180, 1)):
        box = F.Setup.box(nx, ny, 4, 4, 1e-3)
        need = box.footprint()
        buf = _DeviceBuffer(need)
        plan = F.Plan.in_memory(box, gpu_device, buf.ptr, need)
        try:
            plan.set_option("block", 4)
            assert plan.info("block") == block
            plan.run(4)
            plan.sync()
        finally:
            plan.close()
            buf.free()


@pytest.mark.parametrize("ny", [66, 133, 300, 3300])
@pytest.mark.parametrize("jcut", [0, 9, 64, 500])
def test_rc_candidates(gpu_device, ny, jcut):
    """The RC maximum over row 0 and rows jcut .. ny-3 (none past the grid),
    the edge carried over launches of 8, 3 and the rest, with a NaN at row 0 of
    one probe column."""
    rng = np.random.default_rng(ny + jcut)
    p = random_problem(rng, nx=140, ny=ny, npml=5, nsteps=30, table=True)
    p.src_table = p.src_table * 50
    p.rc_imax = np.array([50, 80, 101], np.int32)
    p.rc_i = p.rc_imax + np.int32(2)
    p.rc_jcut, p.rc_level, p.rc_edge0 = jcut, 0.07, 1e-4
    ez = np.zeros((ny, 140), np.float32)
    ez[0, 80] = np.nan  # a ring cell: never updated
    ref = Oracle(p, 32)
    ref.write_field(F.EZ, ez)
    ref.run(p.nsteps)
    with F.Plan(p, gpu_device) as plan:
        plan.write_field(F.EZ, ez)
        for n in (8, 3, 19):
            plan.run(n)
        assert np.array_equal(plan.read_rc(), np.asarray(ref.read_rc()))


@pytest.mark.parametrize("nx,ny", [(64, 33), (100, 40), (129, 70), (256, 31), (700, 90)])
def test_field_and_psi_round_trip(gpu_device, nx, ny):
    """Fields and psi strips written and read back through rows that are and
    are not contiguous on the device, Hx and Hy with their shorter sides."""
    P = 5
    rng = np.random.default_rng(nx + ny)
    p = random_problem(rng, nx=nx, ny=ny, npml=P, nsteps=4, table=False)
    with F.Plan(p, gpu_device) as plan:
        for which in (F.EZ, F.HX, F.HY, F.JZ):
            v = rng.standard_normal(plan.read_field(which).shape).astype(np.float32)
            plan.write_field(which, v)
            assert np.array_equal(_bits(plan.read_field(which)), _bits(v)), which
        for which in (F.PSI_HXY, F.PSI_EZY, F.PSI_HYX, F.PSI_EZX):
            v = rng.standard_normal(plan.read_psi(which).shape).astype(np.float32)
            plan.write_psi(which, v)
            assert np.array_equal(_bits(plan.read_psi(which)), _bits(v)), which
        # both buffer sets took the values: a step reads one and writes the other
        ref = Oracle(p, 32)
        for which in (F.EZ, F.HX, F.HY, F.JZ):
            ref.write_field(which, plan.read_field(which))
        for which in (F.PSI_HXY, F.PSI_EZY, F.PSI_HYX, F.PSI_EZX):
            ref.write_psi(which, plan.read_psi(which))
        ref.run(4)
        for n in (1, 3):
            plan.run(n)
        want = all_state(ref, P)
        got = all_state(plan, P)
    for k in want:
        assert np.array_equal(_bits(want[k]), _bits(got[k])), k


def _pool_check(pool, ids, probs, label):
    for sid, p in zip(ids, probs):
        ref = Oracle(p, 32, threads=4)
        ref.run(p.nsteps)
        det, comp = pool.read_detectors(sid)
        rdet, rcomp = ref.read_detectors()
        assert np.array_equal(_bits(det), _bits(rdet)) and np.array_equal(_bits(comp), _bits(rcomp)), (label, sid)
        for which in (F.EZ, F.HX, F.HY, F.JZ):
            assert np.array_equal(_bits(pool.read_field(sid, which)), _bits(ref.read_field(which))), (label, sid, which)
        if p.line_size:
            assert np.array_equal(_bits(pool.read_line(sid)), _bits(ref.read_line())), (label, sid)


@pytest.mark.parametrize("table,chunk", [(False, 4), (True, 4), (False, 0)])
def test_pool_block_form(gpu_device, table, chunk):
    """Uneven shots through the block form, with graphs and without: tails of
    every length, shots that join, end and leave between launches (the list
    and the captured grid change), the form switched off and on mid-run."""
    rng = np.random.default_rng(300 + table)
    probs = []
    for k in range(8):
        p = random_problem(rng, nx=int(rng.integers(40, 300)), ny=int(rng.integers(40, 260)),
                           npml=int(rng.choice([0, 5, 12])), nsteps=(33, 40, 47, 26, 64, 71, 35, 58)[k], table=table)
        if k == 2:
            p.line_size, p.line_i0, p.line_j, p.line_begin, p.line_end = 20, 5, 20, 2, 30
        probs.append(p)
    with F.Pool(gpu_device, graph_chunk=chunk) as pool:
        ids = [pool.add(p) for p in probs[:4]]
        assert pool.info("block") == 1
        pool.step(2)
        ids += [pool.add(p) for p in probs[4:6]]
        pool.step(2)
        pool.set_option("block", 0)
        pool.step(1)
        pool.set_option("block", 1)
        pool.step(1)
        pool.sync()
        _pool_check(pool, ids[3:4], probs[3:4], "ended early")
        pool.remove(ids[3])
        ids[3] = pool.add(probs[6])  # the slot comes back
        ids.append(pool.add(probs[7]))
        while pool.info("running") > 0:
            pool.step(max(chunk, 1))
        pool.sync()
        _pool_check(pool, ids, probs[:3] + [probs[6]] + probs[4:6] + [probs[7]], f"table={table} chunk={chunk}")
        if chunk:
            assert pool.info("graph_replays") > 0
        pool.set_option("wg_per_cu", 3)  # an option of the streaming form
        assert pool.info("block") == 0


def test_block_form_repeats(gpu_device):
    """Many runs of the same small table-medium shots, block form, against the
    streaming form's bits: a wave that reads its neighbour's edge row before it
    has arrived (a barrier without the wait for the LDS writes before it) shows
    only now and then."""
    rng = np.random.default_rng(13)
    probs = [random_problem(rng, nx=nx, ny=ny, npml=12, nsteps=320, table=True)
             for nx, ny in ((221, 198), (221, 294), (170, 282), (261, 408))]

    def run(block):
        with F.Pool(gpu_device) as pool:
            pool.set_option("block", block)
            ids = [pool.add(p) for p in probs]
            while pool.info("running") > 0:
                pool.step(8)
            return [pool.read_field(sid, F.EZ) for sid in ids]

    want = run(0)
    for k in range(60):
        for s, (a, b) in enumerate(zip(want, run(1))):
            assert np.array_equal(_bits(a), _bits(b)), f"run {k} shot {s}"
