"""Steps that no block can hold together (-m gpu): with more than 2048
hypercolumns the tuned plans run them, blocks run the others; against the
oracle, with the launches counted."""

import numpy as np
import pytest

import oracle as O
from gsbn_amd import Solver, configs
from helpers import compare_state

pytestmark = pytest.mark.gpu


def _spec(H):
    """A stimulus row of its own for every step, then windows of 20 steps, then
    single ones again."""
    spec = configs.recall_net(4, 3, 4, 20, 0, 20, 0.5, seed=2, name="alone")
    rng = np.random.Generator(np.random.Philox(2))
    spec.pops[0].hcu, spec.pops[0].mcu = H, 3
    ii, di, C = configs.sparse_conn_arrays(rng, H, 3, 20.0 / H)
    spec.conn, spec.conn_arrays = [[]], [(ii, di)]
    spec.projs[0].slot_num = float(C)
    spec.stim = rng.integers(0, 3, (5, H)).astype(np.uint32)
    spec.mask = np.ones((1, H), np.float32)
    at = [configs.step_time(t, spec.dt) for t in range(0, 200)]
    spec.modes = [configs.ModeSpec(at[t], at[t + n * k], time_step=n, begin_lgidx_id=0, lgidx_step=1,
                                   begin_wmask_id=0, wmask_step=0, prn=1.0)
                  for t, n, k in [(4 * i, 1, 4) for i in range(10)] + [(40, 20, 3)] +
                  [(100 + 4 * i, 1, 4) for i in range(10)]]
    return spec


@pytest.mark.parametrize("H,alone", [(2049, True), (2048, False)])
def test_steps_alone(tmp_path, H, alone):
    spec = _spec(H)
    gpu = Solver(configs.write(spec, str(tmp_path)))
    configs.apply_conn_arrays(gpu, spec)
    ora = O.OracleNet(spec)
    gpu.step(3)  # a launch of each kind is counted from here
    gpu.timing(-1, collect=False)
    gpu.timing((1 << 0) | (1 << 6), collect=False)
    gpu.step(37)
    single = gpu.timing(1 << 0 | 1 << 6)[0].copy()
    gpu.step(60)
    both = gpu.timing(1 << 0 | 1 << 6)[0].copy()
    gpu.step(39)
    last = gpu.timing(0)[0]
    gpu.timing(-1, collect=False)
    for _ in range(139):
        ora.step()
    assert not compare_state(gpu, ora, spec)
    # kind 0: population launches of the split plans; 6: blocks (and chained steps)
    steps = single[0] + single[6]
    assert steps == 37
    assert both[0] + both[6] - steps <= 24  # 60 steps, blocks of three
    if not alone:
        assert single[0] == 0 and last[0] == both[0]
    gpu.close()
    # the kinds apart: without the chained plan, kind 6 is the blocks'
    if alone:
        spec.chained_step = -1
        gpu = Solver(configs.write(spec, str(tmp_path)))
        configs.apply_conn_arrays(gpu, spec)
        gpu.step(3)
        gpu.timing(-1, collect=False)
        gpu.timing((1 << 0) | (1 << 6), collect=False)
        gpu.step(37)
        n = gpu.timing(0)[0]
        gpu.timing(-1, collect=False)
        assert n[0] >= 36 and n[6] <= 1
        gpu.close()
