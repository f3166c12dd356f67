"""Two solvers open in one program (-m gpu): the results of one are read on its
own stream, whatever the other one did last, and after the other is closed."""

import numpy as np
import pytest

import gsbn_amd
from gsbn_amd import Solver, configs

pytestmark = pytest.mark.gpu

STEPS = 560  # eleven windows scored, the schedule not at its end


def _spec(nets):
    """Recall windows of 50 steps, one after the other (no learning); of many
    networks, so that the device is behind the host when a call returns."""
    spec = configs.batched_nets(nets, 12, 50, 0, 50, 0, hcu_range=(8, 40), mcu_range=(16, 90),
                                seed=7)
    spec.modes = [m for m in spec.modes if m.prn == 0.0]
    (mode,) = spec.modes
    shift = mode.begin_time - configs.step_time(0, spec.dt)
    mode.begin_time -= shift
    mode.end_time -= shift
    return spec


def _solver(spec, path):
    path.mkdir(exist_ok=True)
    s = Solver(configs.write(spec, str(path)))
    configs.apply_conn_arrays(s, spec)
    return s


def _log(path):
    (f,) = sorted(path.rglob("check_result.txt"))
    return f.read_text().splitlines()


@pytest.mark.parametrize("closed", [False, True])
def test_scores_are_read_on_the_solvers_own_stream(tmp_path, closed):
    spec = _spec(150)
    gsbn_amd.release_memory()  # no earlier run's scores in a's arrays
    a = _solver(spec, tmp_path / "a")
    b = _solver(_spec(2), tmp_path / "b")
    # (the simulated time is the program's, shared by its solvers; b only has
    # to be the one used last)
    a.step(STEPS)
    b.sync()
    if closed:
        b.close()
    got, lines = a.check(), _log(tmp_path / "a")
    if not closed:
        b.close()
    a.close()
    alone = _solver(spec, tmp_path / "c")
    alone.step(STEPS)
    alone.sync()
    want = alone.check()
    assert want[1] == 11
    assert got[:2] == want[:2] and np.array_equal(got[2], want[2])
    assert lines == _log(tmp_path / "c")
    alone.close()


def test_state_is_read_on_the_solvers_own_stream(tmp_path):
    spec = _spec(150)
    names = ("spike_3", "dsup_149", "wij_0", "tij_1", "pj_0")
    gsbn_amd.release_memory()
    a = _solver(spec, tmp_path / "a")
    b = _solver(_spec(2), tmp_path / "b")
    a.step(STEPS)
    b.sync()
    got = {n: a.vector(n) for n in names}
    b.close()
    a.close()
    alone = _solver(spec, tmp_path / "c")
    alone.step(STEPS)
    for n, w in got.items():
        assert alone.vector(n).tobytes() == w.tobytes(), n
    alone.close()
