"""The choice of the step plan (-m gpu) where a learning-rate change is recorded
before the choice is made: it is made all the same, for the steps with recorded
changes and, after the log is emptied, for those without."""

import pytest

import oracle as O
from gsbn_amd import Solver, configs
from helpers import compare_state

pytestmark = pytest.mark.gpu


def _spec(H=10, M=10):
    """One change of the learning rate at step 31, then one rate."""
    spec = configs.recall_net(H, M, 3, 30, 0, 30, 0.4, name="tune")
    first = spec.modes[0]
    rest = configs.ModeSpec(**{**first.__dict__})
    first.end_time = configs.step_time(30, spec.dt)
    rest.begin_time, rest.end_time = first.end_time, configs.step_time(900, spec.dt)
    rest.time_step, rest.begin_lgidx_id, rest.lgidx_step, rest.prn = 870, 1, 0, 0.5
    spec.modes = [first, rest]
    spec.deferred_sweeps = 1
    return spec


@pytest.mark.parametrize("batch", [False, True])
def test_tuning_ends_with_a_change_recorded(tmp_path, batch):
    spec = _spec()
    if batch:
        two = configs.batched_nets(3, 3, 30, 0, 30, 0, hcu_range=(4, 8), mcu_range=(5, 12), seed=3)
        two.modes, two.deferred_sweeps = spec.modes, 1
        spec = two
    gpu = Solver(configs.write(spec, str(tmp_path)))
    configs.apply_conn_arrays(gpu, spec)
    ora = O.OracleNet(spec)
    seen = []
    for t in range(700):
        gpu.step(1)
        ora.step()
        if t == 350:
            assert gpu.glob("plan-tuned") == 1 and gpu.glob("rowcol-parts") != -2
            gpu.vector("wij_0")  # the log is emptied
            if batch:
                gpu.vector("wij_1"), gpu.vector("wij_2")
        if t in (352, 699):
            seen.append(gpu.glob("plan-tuned"))
    assert seen == [0, 1]
    assert gpu.glob("deferred-sweeps") == 1 and gpu.work()[4] == 2
    assert not compare_state(gpu, ora, spec)
    gpu.close()


def test_a_choice_made_before_serves_the_steps_after(tmp_path):
    spec = _spec()
    spec.modes[0].end_time = spec.modes[1].begin_time = configs.step_time(300, spec.dt)
    spec.modes[0].time_step = 300
    gpu = Solver(configs.write(spec, str(tmp_path)))
    ora = O.OracleNet(spec)
    for t in range(500):
        gpu.step(1)
        ora.step()
        if t in (290, 499):
            assert gpu.glob("plan-tuned") == 1
    assert not compare_state(gpu, ora, spec)
    gpu.close()
