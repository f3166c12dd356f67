"""Rings of column kicks as deep as the steps need (-m gpu): shallow ones in
single steps, deep ones from the first block or recorded sweep on, with the
kicks that are pending then, and the depth in use reported; against the oracle."""

import pytest

import oracle as O
from gsbn_amd import Solver, configs
from helpers import compare_state

pytestmark = pytest.mark.gpu


def _spec(k, batch=False, **net):
    if batch:
        spec = configs.batched_nets(4, 3, 40, 5, 20, 10, hcu_range=(3, 9), mcu_range=(5, 70), seed=6)
    else:
        spec = configs.recall_net(8, 9, 3, 40, 5, 20, 0.4, reset=10, name="ring")
    for p in spec.pops:
        p.maxfq = 700.0  # rings fill and are walked
    for key, v in k.items():
        setattr(spec, key, v)
    return spec


@pytest.mark.parametrize("batch", [False, True])
@pytest.mark.parametrize("k,single,blocks,changed", [
    (dict(), 0, 64, 64),                       # 0: the default, 8 or 16
    (dict(block_step=0), 0, 0, 0),
    (dict(block_step=0, deferred_sweeps=1), 0, 0, 64),
    (dict(block_step=0, deferred_sweeps=1, trace_precision="bf16"), 0, 0, 64),
    (dict(chained_step=-1), 0, 64, 64),
    (dict(deferred_columns=4), 4, 4, 4),
    (dict(deferred_columns=32, deferred_sweeps=1), 32, 32, 32),
])
def test_depth(tmp_path, batch, k, single, blocks, changed):
    spec = _spec(k, batch)
    base = 16 if batch else 8
    gpu = Solver(configs.write(spec, str(tmp_path)))
    configs.apply_conn_arrays(gpu, spec)
    ora = O.OracleNet(spec)
    f = 0

    def run(n, call):
        nonlocal f
        for _ in range(0, n, call):
            gpu.step(call)
        for _ in range(n):
            if f >= 0:
                f = ora.step()

    def depth():
        assert gpu.glob("deferred-ring") == gpu.glob("deferred-columns")
        return gpu.glob("deferred-columns")

    run(90, 1)
    assert depth() == (single or base)
    run(30, 10)  # the training ends at 135
    assert depth() == (blocks or base)
    assert not compare_state(gpu, ora, spec)
    run(30, 1)   # the rate changes
    assert depth() == (changed or base)
    while f >= 0:
        run(21, 7)
    assert not compare_state(gpu, ora, spec)
    gpu.close()


def test_pending_kicks_of_every_count(tmp_path):
    """The rings deepen after every number of steps, with one kick to a full
    ring pending per unit."""
    for n in range(1, 30):
        spec = _spec(dict())
        (tmp_path / str(n)).mkdir()
        gpu = Solver(configs.write(spec, str(tmp_path / str(n))))
        ora = O.OracleNet(spec)
        for _ in range(n):
            gpu.step(1)
        assert gpu.glob("deferred-columns") == 8
        gpu.step(41)
        assert gpu.glob("deferred-columns") == 64
        for _ in range(n + 41):
            ora.step()
        assert not compare_state(gpu, ora, spec), n
        gpu.close()
