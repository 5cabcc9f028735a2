"""The streaming form of the step kernels on the grids and shots that take the
block form by themselves: tests of other files that leave the form to the
library, run again with it switched off in every plan and pool they make."""

from __future__ import annotations

import pytest

import fdtd2d_amd as F

from test_gpu_block import test_rc_candidates  # noqa: F401
from test_gpu_configs import test_batch_mix_first_16_shots  # noqa: F401
from test_gpu_driver import (  # noqa: F401
    test_shipped_settings_on_gpu_match_oracle,
    test_shipped_settings_rc_lines_match_oracle,
)
from test_gpu_parity import (  # noqa: F401
    test_jz_written_where_no_plasma,
    test_nonuniform_den_inside,
    test_rc_lines_match_oracle,
    test_resume_equals_single_run,
    test_write_field_initial_state,
)
from test_gpu_pool import test_pool_budget_admission_and_slot_reuse, test_pool_processing_lines  # noqa: F401
from test_zz_no_alloc import test_create_in_matches_create  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def streaming(monkeypatch):
    """Switches the block form off in every plan and pool the test makes; each
    run and step checks that it is."""

    def off(sim):
        sim.set_option("block", 0)
        assert sim.info("block") == 0
        made.append(sim)

    def checked(method):
        def call(self, *args):
            assert self.info("block") == 0
            return method(self, *args)

        return call

    made = []
    plan_init, plan_in, pool_init = F.Plan.__init__, F.Plan.in_memory.__func__, F.Pool.__init__

    def new_plan(self, *args, **kwargs):
        plan_init(self, *args, **kwargs)
        off(self)

    def new_plan_in(cls, *args, **kwargs):
        plan = plan_in(cls, *args, **kwargs)
        off(plan)
        return plan

    def new_pool(self, *args, **kwargs):
        pool_init(self, *args, **kwargs)
        off(self)

    monkeypatch.setattr(F.Plan, "__init__", new_plan)
    monkeypatch.setattr(F.Plan, "in_memory", classmethod(new_plan_in))
    monkeypatch.setattr(F.Pool, "__init__", new_pool)
    monkeypatch.setattr(F.Plan, "run", checked(F.Plan.run))
    monkeypatch.setattr(F.Pool, "step", checked(F.Pool.step))
    yield
    assert made
