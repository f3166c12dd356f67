"""The log of recorded sweeps (-m gpu): more changes than it holds, and the
synapse updates of a sweep counted when they are made; against the oracle."""

import pytest

import oracle as O
from gsbn_amd import Solver, configs
from helpers import compare_state

pytestmark = pytest.mark.gpu

CUES = 15


def _spec(k):
    """Two changes per cue after the training: 31 with the first step's."""
    spec = configs.recall_net(6, 7, CUES, 8, 0, 7, 0.4, reset=5, name="log")
    for key, v in k.items():
        setattr(spec, key, v)
    return spec


@pytest.mark.parametrize("k", [dict(), dict(trace_precision="fp16"), dict(block_step=0),
                               dict(rowcol_parts=2), dict(deferred_columns=8)])
@pytest.mark.parametrize("defer", [1, 0])
@pytest.mark.parametrize("call", [1, 6])
def test_more_changes_than_the_log_holds(tmp_path, k, defer, call):
    spec = _spec(dict(k, deferred_sweeps=defer))
    gpu = Solver(configs.write(spec, str(tmp_path)))
    ora = O.OracleNet(spec)
    one = 6 * 5 * 7 * 7  # synapses: H x (H - 1) M slots x M
    f, seen = 0, set()
    while f >= 0:
        for _ in range(call):
            f = ora.step() if f >= 0 else f
        gpu.step(call)
        w = gpu.work()
        assert w[2] % one == 0
        seen.add((int(w[4]), int(w[2]) // one))
    assert gpu.glob("deferred-sweeps") == defer
    assert (1 + 2 * CUES, 1 + 2 * CUES) in seen
    if defer:
        # the first change has nothing to sweep; the next 16 fill the log, which
        # is applied at the 18th change and at the end
        assert sorted({s for _, s in seen}) == [1, 17, 31]
        assert all(s == 1 for c, s in seen if c <= 17)
    else:
        assert all(c == s for c, s in seen)
    assert not compare_state(gpu, ora, spec)
    gpu.close()
