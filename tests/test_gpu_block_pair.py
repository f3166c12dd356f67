"""Block steps of populations connected to each other (-m gpu): two in a loop,
and three in a ring, each with one incoming and one outgoing projection, of
different sizes and delays, up to a spike of a unit in every step (the rings
then fill between two walks); against the oracle, bit for bit."""

import numpy as np
import pytest

import oracle as O
from gsbn_amd import Solver, configs
from helpers import compare_state

pytestmark = pytest.mark.gpu


def _conn(rng, src, dest, C, delays):
    """C slots per destination hypercolumn, the last one empty."""
    ii = np.full((dest[0], C), -1, np.int32)
    for h in range(dest[0]):
        ii[h, :C - 1] = np.sort(rng.permutation(src[0] * src[1])[:C - 1])
    di = np.where(ii >= 0, rng.integers(delays[0], delays[1] + 1, ii.shape), 0).astype(np.int32)
    return ii.reshape(-1), di.reshape(-1)


def _spec(sizes, delays, seed, maxfq=700.0, **k):
    rng = np.random.Generator(np.random.Philox(seed))
    spec = configs.recall_net(4, 3, 3, 80, 5, 50, 0.5, seed=seed, reset=9, name="pair")
    n = len(sizes)
    spec.pops = [configs.PopSpec(hcu=H, mcu=M, wtagain=4.0, wgain=8.0, snoise=0.1, maxfq=maxfq)
                 for H, M in sizes]
    spec.projs, spec.conn_arrays, spec.conn = [], [], [[] for _ in range(n)]
    for i in range(n):  # population i feeds i + 1
        d = (i + 1) % n
        C = min(sizes[i][0] * sizes[i][1], 41)
        spec.projs.append(configs.ProjSpec(src=i, dest=d, tauzi=0.01, tauzj=0.01, taue=0.02,
                                           taup=1.0, slot_num=float(C)))
        spec.conn_arrays.append(_conn(rng, sizes[i], sizes[d], C, delays[i]))
    units = sum(H for H, _ in sizes)
    rows = spec.stim.shape[0]
    spec.stim = np.concatenate([rng.integers(0, M, (rows, H)) for H, M in sizes], 1).astype(np.uint32)
    spec.mask = (rng.random((spec.mask.shape[0], units)) < 0.7).astype(np.float32)
    spec.mask[0] = 0.0  # the training, without recurrent support
    spec.block_step = 1
    for key, v in k.items():
        setattr(spec, key, v)
    return spec


@pytest.mark.parametrize("sizes,delays", [
    (((5, 9), (7, 4)), ((1, 1), (1, 1))),
    (((6, 70), (9, 20)), ((1, 4), (3, 6))),
    (((12, 5), (3, 64), (20, 8)), ((2, 2), (1, 5), (7, 31))),
])
@pytest.mark.parametrize("k", [dict(), dict(deferred_sweeps=1), dict(trace_precision="fp16"),
                               dict(maxfq=1000.0), dict(maxfq=1000.0, deferred_sweeps=1)])
@pytest.mark.parametrize("chunk", [10**9, 7])
def test_populations_in_a_ring(tmp_path, sizes, delays, k, chunk):
    spec = _spec(sizes, delays, 4, **k)
    gpu = Solver(configs.write(spec, str(tmp_path)))
    configs.apply_conn_arrays(gpu, spec)
    ora = O.OracleNet(spec)
    f, spikes = 0, 0
    while f >= 0:
        n = 0
        while f >= 0 and n < chunk:
            f = ora.step()
            n += 1
            spikes += int(ora.vector("spike_0").sum()) if f >= 0 else 0
        gpu.step(n)
        if f >= 0:
            for i in range(len(sizes)):
                assert gpu.vector("spike_%d" % i).tobytes() == ora.vector("spike_%d" % i).tobytes()
    assert gpu.glob("block-step") == 1
    assert spikes > 100
    assert not compare_state(gpu, ora, spec)
    gpu.close()
