"""The recall's one-wave-per-(HCU, cue) kernel (-m gpu) at the edges of its
paths: units per lane, launches of several steps, up to and beyond 64 active
sources, several delays and slots per source.

* mfma: every step's spikes equal those of the dense product (which a run
  that times the product uses), for weights whose sums are exact and weights
  of mixed magnitude, whose sums round;
* exact: every step's spikes equal the oracle's, cue by cue.
"""

import numpy as np
import pytest

import oracle as O
from gsbn_amd import configs
from gsbn_amd import recall as R

pytestmark = pytest.mark.gpu


def _net(H, M, C, maxfq):
    pop = configs.PopSpec(hcu=H, mcu=M, wgain=2.0, snoise=0.5, maxfq=maxfq)
    proj = configs.ProjSpec(src=0, dest=0, tauzi=0.01, tauzj=0.01, taue=0.02, taup=1.0,
                            slot_num=float(C))
    return configs.NetSpec(dt=0.001, pops=[pop], projs=[proj], modes=[], stim=np.zeros((0, H)),
                           mask=np.zeros((0, H)), conn=[[]])


def _cues(rng, H, M, B):
    clamp = np.where(rng.random((B, H)) < 0.4, rng.integers(0, M, (B, H)), -1).astype(np.int16)
    return clamp, (clamp < 0).astype(np.float32)


@pytest.mark.parametrize("H,M,B,maxfq,delay,mixed", [
    (3, 5, 1, 100.0, 1, False), (10, 64, 9, 500.0, 1, True), (7, 65, 17, 500.0, 3, True),
    (9, 128, 8, 300.0, 1, True), (4, 200, 11, 500.0, 2, True), (180, 12, 10, 500.0, 1, True),
    (40, 30, 33, 100.0, 1, False)])
def test_mfma_equals_the_dense_product(H, M, B, maxfq, delay, mixed):
    rng = np.random.default_rng(H * 1000 + M)
    N, C = H * M, max(1, (H * M) // 2)
    ii = np.full((H, C), -1, np.int32)
    for h in range(H):
        ii[h, :C - 1] = np.sort(rng.permutation(N)[:C - 1])
    ii = ii.reshape(-1)
    di = np.where(ii >= 0, delay, 0).astype(np.int32)
    wij = rng.normal(0, 0.3, (H * C, M)).astype(np.float32)
    if mixed:
        wij *= np.exp2(rng.integers(-20, 3, wij.shape)).astype(np.float32)
        wij[rng.random(wij.shape) < 0.1] = 0.0
    bj = rng.normal(-1, 0.3, N).astype(np.float32)
    clamp, wmask = _cues(rng, H, M, B)
    rc = R.Recall(H, M, C, ii, di, wij, bj, R.population_params(_net(H, M, C, maxfq)), B, R.MFMA, 5)
    steps = 23
    idx, cnt, ras, _ = rc.run(clamp, wmask, steps, count_from=4, raster=True)
    didx, dcnt, dras, ms = rc.run(clamp, wmask, steps, count_from=4, raster=True, time_support=True)
    assert ms > 0
    assert np.array_equal(ras, dras)
    assert np.array_equal(idx, didx) and np.array_equal(cnt, dcnt)
    rc.close()


@pytest.mark.parametrize("H,M,B,maxfq,delays,repeat", [
    (3, 1, 2, 100.0, 1, 1), (10, 64, 3, 500.0, 1, 1), (7, 65, 3, 500.0, 5, 1),
    (5, 130, 3, 900.0, 1, 3), (4, 256, 2, 900.0, 31, 2), (90, 6, 2, 1000.0, 1, 1)])
def test_exact_equals_the_oracle(H, M, B, maxfq, delays, repeat):
    rng = np.random.default_rng(H * 1000 + M)
    N = H * M
    C = N  # a projection has at most one slot per source unit
    # sources up to `repeat` times among the slots, in no order, some slots empty
    ii = np.stack([rng.permutation(np.tile(np.arange(N), repeat))[:C] for _ in range(H)])
    ii = np.where(rng.random(ii.shape) < 0.05, -1, ii).astype(np.int32).reshape(-1)
    di = np.where(ii >= 0, rng.integers(1, delays + 1, ii.size), 0).astype(np.int32)
    wij = rng.normal(0, 0.3, (H * C, M)).astype(np.float32)
    bj = rng.normal(-1, 0.3, N).astype(np.float32)
    spec = _net(H, M, C, maxfq)
    clamp, wmask = _cues(rng, H, M, B)
    steps = 40
    rc = R.Recall(H, M, C, ii, di, wij.reshape(-1), bj, R.population_params(spec), B, R.EXACT, 77)
    idx, cnt, ras, _ = rc.run(clamp, wmask, steps, count_from=0, raster=True)
    rc.close()
    for b in range(B):
        net = O.OracleNet(R.oracle_recall_spec(spec, clamp[b], wmask[b], steps, 77 + b, ii, di))
        net.write("wij_0", wij.reshape(-1))
        net.write("bj_0", bj)
        counts = np.zeros(N, np.int64)
        for t in range(steps):
            net.step()
            want = net.vector("spike_0")
            assert np.array_equal(ras[t, b], want), (b, t)
            counts += want
        c = counts.reshape(H, M)
        assert np.array_equal(cnt[b], c.max(axis=1))
        assert np.array_equal(idx[b], np.where(c.max(axis=1) > 0, c.argmax(axis=1), -1))
