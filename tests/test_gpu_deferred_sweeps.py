"""Deferred sweeps (-m gpu): learning-rate changes recorded and applied later
leave the state of the sweeps, bit for bit against the oracle, with more
changes than the log holds, reads of the state between them, in every trace
form, row/column plan and ring depth, in batches, and over a resume."""

import numpy as np
import pytest

import oracle as O
from gsbn_amd import Solver, configs
from helpers import compare_state, run_lockstep

pytestmark = pytest.mark.gpu


def _spec(hcu=6, mcu=7, n_pat=3, **k):
    """Short windows, so that the learning rate switches often (two changes
    per cue), with a learning rate of every kind: 1, negligible, 0."""
    spec = configs.recall_net(hcu, mcu, n_pat, 12, 5, 9, 0.4, reset=6, name="ds")
    # a second round of training and recall on the weights of the first
    t = int(round(spec.modes[-1].end_time / spec.dt - 0.5))
    again = []
    for m in spec.modes:
        c = configs.ModeSpec(**{**m.__dict__})
        c.begin_time += t * spec.dt
        c.end_time += t * spec.dt
        again.append(c)
    spec.modes = spec.modes + again + [
        configs.ModeSpec(**{**m.__dict__, "begin_time": m.begin_time + 2 * t * spec.dt,
                            "end_time": m.end_time + 2 * t * spec.dt}) for m in spec.modes]
    spec.deferred_sweeps = 1
    for key, v in k.items():
        setattr(spec, key, v)
    return spec


@pytest.mark.parametrize("k", [
    dict(), dict(trace_precision="bf16"), dict(trace_precision="fp16"),
    dict(rowcol_parts=1), dict(rowcol_parts=3, deferred_columns=2), dict(deferred_columns=64),
    dict(deferred_sweeps=0), dict(chained_step=1), dict(exchange_direct=False)])
def test_state_equals_the_oracle(tmp_path, k):
    spec = _spec(**k)
    gpu, ora, diverged, steps = run_lockstep(spec, tmp_path)
    assert diverged is None
    assert gpu.glob("deferred-sweeps") == (0 if "deferred_sweeps" in k or "chained_step" in k else 1)
    assert gpu.work()[4] > 16 or steps > 100
    assert not compare_state(gpu, ora, spec)
    gpu.close()


def test_reads_between_the_changes(tmp_path):
    spec = _spec(trace_precision="fp16")
    gpu, ora, diverged, _ = run_lockstep(spec, tmp_path, check_every=13)
    assert diverged is None
    gpu.close()


def test_a_host_write_between_the_changes(tmp_path):
    spec = _spec()
    gpu = Solver(configs.write(spec, str(tmp_path)))
    ora = O.OracleNet(spec)
    for t in range(200):
        if t == 83:
            for s in (gpu, ora):
                w = s.vector("pij_0")
                s.write("pij_0", (w * np.float32(1.5)).astype(np.float32))
        gpu.step(1)
        ora.step()
    assert not compare_state(gpu, ora, spec)
    gpu.close()


@pytest.mark.parametrize("k", [dict(), dict(rowcol_wave=1), dict(rowcol_wave=2),
                               dict(rowcol_graded=2), dict(rowcol_parts=2, pop_wave=0),
                               dict(trace_precision="bf16", rowcol_wave=1, ovf_keep=1)])
def test_batches(tmp_path, k):
    spec = configs.batched_nets(5, 3, 12, 4, 9, 6, hcu_range=(3, 9), mcu_range=(5, 70),
                                probs=(0.4, 0.9), seed=4)
    spec.deferred_sweeps = 1
    for key, v in k.items():
        setattr(spec, key, v)
    gpu = Solver(configs.write(spec, str(tmp_path)))
    configs.apply_conn_arrays(gpu, spec)
    ora = O.OracleNet(spec)
    f, t = 0, 0
    while f >= 0:
        gpu.step(1)
        f = ora.step()
        t += 1
        if t == 70:  # one network's state is read: its log is applied alone
            assert np.array_equal(gpu.vector("wij_1").view(np.uint32),
                                  ora.vector("wij_1").view(np.uint32))
    assert not compare_state(gpu, ora, spec)
    gpu.close()


def test_resume_with_changes_recorded(tmp_path):
    spec = _spec()
    path = configs.write(spec, str(tmp_path))
    a = Solver(path)
    a.step(100)
    a.snapshot(str(tmp_path / "s.bin"))
    a.step(120)
    want = {n: a.vector(n) for n in ("wij_0", "pij_0", "eij_0", "tij_0", "pi_0", "ti_0", "spike_0")}
    a.close()
    b = Solver(path, str(tmp_path / "s.bin"))
    b.step(120)
    for n, w in want.items():
        assert b.vector(n).tobytes() == w.tobytes(), n
    b.close()
