"""The step kernels' form in the tuners and the shape cache, on the CPU: fakes
stand in for the device pool and plan, and trials are scored from their
options, so the tests check which shapes were tried, kept and looked up."""

from __future__ import annotations

import json

import pytest

from fdtd2d_amd import batch, tuning
from fdtd2d_amd.tuning import SHIPPED, ShapeCache, form_key, is_block_key, key_distance, mix_key

STREAM = {"tblock": 8, "cols_per_lane": 2, "band": 64}
BLOCK = {"tblock": 8, "block": 1}


class FakePlan:
    """A plan that is in the block form until a streaming option is set."""

    def __init__(self, block, nsteps=4000):
        self.options = {"tblock": 8, "cols_per_lane": 2, "band": 96, "prefetch": 2}
        self.block, self.n, self.nsteps, self.nx, self.ny = block, 0, nsteps, 1000, 1000

    def set_option(self, name, value):
        if name == "block":
            self.block = int(value)
        else:
            self.options[name] = value
            if name != "tblock":
                self.block = 0

    def info(self, name):
        return {"steps": self.n, "block": self.block, **self.options}[name]

    def run(self, steps):
        self.n += steps

    def sync(self):
        pass


class FakePool(batch.Pool):
    """A pool in the block form while no streaming option is set and its cells
    are under the limit."""

    def __init__(self, cells=5e7):
        self._h = None
        self.options, self.steps, self.cells, self.block = {}, 0, cells, -1

    def set_option(self, name, value):
        if name == "block":
            self.block = int(value)
            return
        self.options[name] = value
        if name != "tblock":
            self.block = 0

    def info(self, name):
        block = self.block if self.block >= 0 else self.cells <= 1.1e8
        return {"cus": 256, "running": 3, "block": int(block), "block_cells_density": 1.1e8, "block_cells_table": 9e7,
                **{"tblock": 8, **self.options}}[name]

    def step(self, n):
        self.steps += n

    def sync(self):
        pass


def _pool_trial(block_gain):
    def trial(pool, launches):
        pool.step(launches)
        return (100.0 + (block_gain if pool.info("block") else 0.0)) * 1e9

    return trial


def test_form_key():
    assert form_key("m1|10:1,11:9", True) == "m1b|10:1,11:9"
    assert form_key("m1b|10:1,11:9", True) == "m1b|10:1,11:9"
    assert form_key("m1b|12x12|P16", False) == form_key("m1|12x12|P16", False) == "m1|12x12|P16"
    assert form_key("", True) == ""
    assert is_block_key("m0+1b|9:10") and not is_block_key("m1|9:10")
    assert key_distance("m1|10:10", "m1b|10:10") == float("inf")


def test_pool_key_follows_the_total_cells():
    """Four shots and a hundred of one mix: the first take the block form."""
    few = [(2048, 2048, 1000, 1)] * 4
    many = [(2048, 2048, 1000, 1)] * 100
    assert mix_key(few) == mix_key(many) == "m1|11:10"
    assert batch.pool_key(FakePool(), few) == "m1b|11:10"
    assert batch.pool_key(FakePool(), many) == "m1|11:10"
    # 22 and 26 shots: 92 and 109 million cells, past the table medium's limit
    assert batch.pool_key(FakePool(), [(2048, 2048, 1000, 0)] * 22) == "m0|11:10"
    assert batch.pool_key(FakePool(), [(2048, 2048, 1000, 1)] * 26) == "m1b|11:10"
    off = FakePool()
    off.set_option("block", 0)
    assert batch.pool_key(off, few) == "m1|11:10"


def test_lookup_passes_over_the_other_form(tmp_path):
    path = tmp_path / "shapes.json"
    path.write_text(json.dumps({"entries": [
        {"kind": "pool", "key": "m1|11:10", "cus": 256, "shape": BLOCK},
        {"kind": "plan", "key": "m1|12x13|P16", "cus": 256, "shape": BLOCK},
        {"kind": "pool", "key": "m1b|10:10", "cus": 256, "shape": BLOCK},
    ]}))
    c = ShapeCache(path, shipped=None)
    for nearest in (False, True):
        assert c.lookup("pool", "m1|11:10", 256, nearest=nearest) == (None, None)
        assert c.lookup("pool", "m1|10:10", 256, nearest=nearest) == (None, None)
        assert c.lookup("pool", "m1b|10:10", 256, nearest=nearest)[0] == BLOCK
    assert c.lookup("plan", "m1|12x13|P16", 256) == (None, None)


def test_shipped_table_keeps_the_forms_apart():
    for e in tuning._load(SHIPPED):
        assert bool(e["shape"].get("block")) == is_block_key(e["key"]), e


def test_plan_shape_takes_the_entry_of_its_form(tmp_path):
    path = tmp_path / "shapes.json"
    path.write_text(json.dumps({"entries": [
        {"kind": "plan", "key": "m1|12x12|P16", "cus": 256, "shape": STREAM},
        {"kind": "plan", "key": "m1b|11x11|P16", "cus": 256, "shape": BLOCK},
    ]}))
    c = ShapeCache(path, shipped=None)
    small = FakePlan(block=1)  # a grid of that bucket in the block form keeps it
    rec = tuning.plan_shape(small, "m1|12x12|P16", 256, c)
    assert rec["shape"] is None and small.info("block") == 1 and rec["key"] == "m1b|12x12|P16"
    large = FakePlan(block=0)
    assert tuning.plan_shape(large, "m1|12x12|P16", 256, c)["shape"] == STREAM and large.options["band"] == 64
    assert tuning.plan_shape(FakePlan(block=1), "m1|11x11|P16", 256, c)["shape"] == BLOCK
    assert tuning.plan_shape(FakePlan(block=0), "m1|11x11|P16", 256, c)["shape"] is None


@pytest.mark.parametrize("gain", [50.0, -50.0])
def test_choose_shape_keeps_the_forms_apart(tmp_path, monkeypatch, gain):
    """What a pool in the block form finds, that form or a streaming shape, is
    stored for such pools only, and the other way round."""
    monkeypatch.setattr(batch, "_trial", _pool_trial(gain))
    c = ShapeCache(tmp_path / "shapes.json", shipped=None)
    small = FakePool()
    rec = batch.choose_shape(small, "m1|11:10", c)
    assert ("block" in rec["shape"]) == (gain > 0) and rec["key"] == "m1b|11:10"
    assert small.info("block") == (1 if gain > 0 else 0)
    large = FakePool(cells=4e8)
    rec = batch.choose_shape(large, "m1|11:10", c)
    assert rec["source"] == "trials" and "block" not in rec["shape"] and large.info("block") == 0
    assert not any("block" in shape for shape, _ in rec["trials"])
    again = FakePool(cells=4e8)
    hit = batch.choose_shape(again, "m1|11:10", c)
    assert hit["trials"] == [] and hit["shape"] == rec["shape"] and again.info("block") == 0
    again = FakePool()
    assert batch.choose_shape(again, "m1|11:10", c)["trials"] == [] and again.info("block") == (1 if gain > 0 else 0)


def _plan_trial(block_rate, stream_rate):
    def trial(plan, launches):
        if plan.n + 8 * launches > plan.nsteps:
            return 0.0
        plan.run(8 * launches)
        return block_rate if plan.info("block") else stream_rate

    return trial


@pytest.mark.parametrize("block_rate,stream_rate,nsteps,block", [
    (5e11, 1e11, 4000, 1),  # the block form wins
    (1e11, 5e11, 4000, 0),  # a streaming shape does
    (5e11, 1e11, 70, 1),    # no steps left for a streaming trial
    (5e11, 1e11, 20, 1),    # nor for any: nothing measured, nothing changed
])
def test_tune_plan_leaves_the_block_form_only_for_a_better_shape(monkeypatch, block_rate, stream_rate, nsteps, block):
    monkeypatch.setattr(tuning, "_plan_trial", _plan_trial(block_rate, stream_rate))
    plan = FakePlan(block=1, nsteps=nsteps)
    rec = tuning.tune_plan(plan)
    assert plan.info("block") == block and ("block" in rec["shape"]) == bool(block)
    assert rec["rate"] == (0.0 if nsteps < 32 else max(block_rate, stream_rate))
    assert plan.n <= nsteps
    # a plan in the streaming form stays there
    plan = FakePlan(block=0, nsteps=nsteps)
    assert "block" not in tuning.tune_plan(plan)["shape"] and plan.info("block") == 0
