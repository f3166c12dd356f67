"""Block step (-m gpu): several steps per launch leave the state of the steps
one by one, bit for bit against the oracle: sizes at the edges of a wave, of
the rows held on chip and of its row list, delays that bound the block,
learning-rate changes inside it, reads, writes and window scores between."""

import numpy as np
import pytest

import oracle as O
from gsbn_amd import Solver, configs
from helpers import compare_state

pytestmark = pytest.mark.gpu


def _spec(H, M, p=0.5, delays=(1, 1), maxfq=100.0, seed=3, train=23, recall=19, **k):
    rng = np.random.Generator(np.random.Philox(seed))
    spec = configs.recall_net(H, M, 1 if M == 1 else 2, train, 7, recall, 0.5, seed=seed, reset=11, name="blk")
    ii, di, C = configs.sparse_conn_arrays(rng, H, M, p)
    di = np.where(ii >= 0, rng.integers(delays[0], delays[1] + 1, ii.size), 0).astype(np.int32)
    spec.conn, spec.conn_arrays = [[]], [(ii, di)]
    spec.projs[0].slot_num = float(C)
    spec.pops[0].maxfq = maxfq
    spec.block_step = 1
    for key, v in k.items():
        setattr(spec, key, v)
    return spec


def _run(spec, tmp_path, chunk=10**9, read=None):
    gpu = Solver(configs.write(spec, str(tmp_path)))
    configs.apply_conn_arrays(gpu, spec)
    ora = O.OracleNet(spec)
    f = 0
    while f >= 0:
        n = 0
        while f >= 0 and n < chunk:
            f = ora.step()
            n += 1
        gpu.step(n)
        if read and f >= 0:
            read(gpu, ora)
    assert gpu.glob("block-step") == 1
    assert not compare_state(gpu, ora, spec)
    c, t, flags = gpu.check()
    assert (c, t) == (ora.check.correct, ora.check.total)
    assert list(flags) == [int(r["ok"]) for r in ora.check.results]
    gpu.close()


@pytest.mark.parametrize("H,M,p,delays,maxfq", [
    (2, 1, 1.0, (1, 1), 400.0),
    (3, 2, 0.9, (2, 31), 900.0),
    (6, 63, 0.4, (1, 4), 300.0),
    (5, 64, 0.5, (6, 9), 300.0),
    (5, 65, 0.5, (4, 4), 300.0),
    (9, 128, 0.2, (1, 2), 500.0),
    (50, 3, 1.0, (1, 1), 1000.0),     # about as many rows as the LDS holds
    (90, 3, 1.0, (3, 3), 1000.0),     # several passes
    (820, 2, 1.0, (1, 1), 1000.0),    # more rows than the list holds, small workgroups
    (300, 3, 0.3, (1, 5), 300.0),
])
def test_sizes(tmp_path, H, M, p, delays, maxfq):
    _run(_spec(H, M, p, delays, maxfq), tmp_path)


@pytest.mark.parametrize("k", [
    dict(trace_precision="bf16"), dict(trace_precision="fp16"), dict(deferred_sweeps=1),
    dict(deferred_sweeps=1, trace_precision="fp16"), dict(deferred_sweeps=1, resident_stimulus=False)])
def test_forms(tmp_path, k):
    _run(_spec(40, 70, 0.3, (1, 3), 900.0, train=97, **k), tmp_path)


@pytest.mark.parametrize("H", [70, 300])
def test_many_rows_and_recorded_changes(tmp_path, H):
    """Rows past those held on chip, in large and small workgroups."""
    _run(_spec(H, 3, 1.0, (1, 2), 1000.0, deferred_sweeps=1), tmp_path)


@pytest.mark.parametrize("chunk", [1, 2, 5, 17])
def test_reads_and_writes_between(tmp_path, chunk):
    def read(gpu, ora):
        read.n += 1
        for n in ("spike_0", "epsc_0", ".ssi_0", "qi_0", "pij_0", "zj2_0")[read.n % 6:][:1]:
            assert gpu.vector(n).tobytes() == ora.vector(n).tobytes(), n
        if read.n % 9 == 4:
            for s in (gpu, ora):
                s.write("pij_0", (s.vector("pij_0") * np.float32(1.25)).astype(np.float32))
                s.write("dsup_0", (s.vector("dsup_0") * np.float32(0.5)).astype(np.float32))
    read.n = 0
    _run(_spec(7, 9, 0.8, (1, 6), 500.0), tmp_path, chunk, read)


@pytest.mark.parametrize("k", [dict(), dict(deferred_sweeps=1, trace_precision="bf16")])
def test_batches(tmp_path, k):
    spec = configs.batched_nets(5, 3, 12, 4, 9, 6, hcu_range=(3, 9), mcu_range=(5, 70),
                                probs=(0.4, 0.9), seed=4)
    spec.block_step = 1
    for key, v in k.items():
        setattr(spec, key, v)
    _run(spec, tmp_path)


def test_calls_of_one_step_between(tmp_path):
    """The tuned plans of single steps (the chained one walks at full rings
    only) and blocks in turn."""
    spec = _spec(6, 8, 0.9, (1, 3), 700.0, train=200)
    spec.block_step = None
    gpu = Solver(configs.write(spec, str(tmp_path)))
    configs.apply_conn_arrays(gpu, spec)
    ora = O.OracleNet(spec)
    f, t = 0, 0
    while f >= 0:
        n = 1 if t % 130 < 90 else 20
        for _ in range(n):
            f = ora.step() if f >= 0 else f
        gpu.step(n)
        t += n
        if t % 130 < 20:
            assert gpu.vector("spike_0").tobytes() == ora.vector("spike_0").tobytes()
    assert gpu.glob("block-step") == 1
    assert not compare_state(gpu, ora, spec)
    gpu.close()


def test_where_it_does_not_apply(tmp_path):
    with pytest.raises(Exception, match="block-step"):
        s = Solver(configs.write(_spec(3, 129), str(tmp_path)))
        s.step(2)
