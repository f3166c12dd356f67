"""Host writes between steps (-m gpu) of the state that pending column kicks and
the queue push depend on: synapse times set back, and slots that get or change
their source.  The kicks of the steps before belong to the synapses as they
were, the push of the last step's spikes to the connectivity as it is; against
the oracle."""

import numpy as np
import pytest

import oracle as O
from gsbn_amd import Solver, configs
from helpers import compare_state

pytestmark = pytest.mark.gpu


def _spec(k):
    spec = configs.recall_net(8, 9, 3, 60, 5, 30, 0.4, reset=10, name="hw")
    rng = np.random.Generator(np.random.Philox(5))
    ii, di, C = configs.sparse_conn_arrays(rng, 8, 9, 0.4)
    spec.conn, spec.conn_arrays = [[]], [(ii, di)]
    spec.projs[0].slot_num = float(C)
    spec.pops[0].maxfq = 400.0
    for key, v in k.items():
        setattr(spec, key, v)
    return spec


def _set_back(s):
    s.write("tij_0", np.maximum(s.vector("tij_0") - 45, 0))


def _new_sources(s):
    ii, di = s.vector("ii_0"), s.vector("di_0")
    free = np.flatnonzero(ii < 0)[::2]
    assert free.size > 3
    ii[free] = 1 + np.arange(free.size, dtype=np.int32) % 7
    di[free] = 2
    s.write("ii_0", ii)
    s.write("di_0", di)


def _other_sources(s):
    """Taken slots whose source or delay changes."""
    ii, di = s.vector("ii_0"), s.vector("di_0")
    taken = np.flatnonzero(ii >= 0)
    ii[taken[::3]] = (ii[taken[::3]] + 11) % 72
    di[taken[1::3]] = 5
    s.write("ii_0", ii)
    s.write("di_0", di)


@pytest.mark.parametrize("write", [_set_back, _new_sources, _other_sources])
@pytest.mark.parametrize("chunk", [1, 50])
@pytest.mark.parametrize("k", [dict(), dict(deferred_columns=4), dict(deferred_columns=64),
                               dict(deferred_columns=0), dict(deferred_sweeps=1),
                               dict(chained_step=1), dict(exchange_direct=False)])
def test_kicks_of_before_a_write(tmp_path, write, chunk, k):
    spec = _spec(k)
    gpu = Solver(configs.write(spec, str(tmp_path)))
    configs.apply_conn_arrays(gpu, spec)
    ora = O.OracleNet(spec)
    for t in range(0, 300, chunk):
        if t in (100, 200):
            write(gpu)
            write(ora)
        gpu.step(chunk)
        for _ in range(chunk):
            ora.step()
        if t == 150:
            assert not compare_state(gpu, ora, spec)
    assert not compare_state(gpu, ora, spec)
    gpu.close()
