"""When a recall handle takes its device memory (-m gpu): the spike matrices of
the dense product with the handle where the product is its path, and otherwise
in the first run that asks for the product's time."""

import gc
import time

import numpy as np
import pytest
import torch

import gsbn_amd
from gsbn_amd import configs
from gsbn_amd import recall as R

pytestmark = pytest.mark.gpu


def _handle(H, M, B):
    rng = np.random.default_rng(3)
    C = H
    ii = np.stack([np.sort(rng.permutation(H * M)[:C]) for _ in range(H)]).astype(np.int32)
    wij = rng.normal(0, 0.3, (H * C, M)).astype(np.float32)
    spec = configs.NetSpec(
        dt=0.001, pops=[configs.PopSpec(hcu=H, mcu=M)],
        projs=[configs.ProjSpec(src=0, dest=0, tauzi=0.01, tauzj=0.01, taue=0.02, taup=1.0,
                                slot_num=float(C))],
        modes=[], stim=np.zeros((0, H)), mask=np.zeros((0, H)), conn=[[]])
    clamp = np.full((B, H), -1, np.int16)
    return R.Recall(H, M, C, ii.reshape(-1), np.ones(H * C, np.int32), wij,
                    np.zeros(H * M, np.float32), R.population_params(spec), B, R.MFMA, 1), \
        (clamp, np.ones((B, H), np.float32))


def _free():
    """Free device memory once it no longer changes: what was given back before
    (by earlier tests, say) is cleared by the driver first and counted late."""
    torch.cuda.synchronize()
    gc.collect()
    last, same = -1, 0
    for _ in range(100):
        now = torch.cuda.mem_get_info()[0]
        same = same + 1 if now == last else 0
        if same == 4:
            break
        last = now
        time.sleep(0.05)
    return now


def _taken(f):
    before = _free()
    r = f()
    return before - _free(), r


# spike matrices: 64 steps x cues rounded to 256 x units rounded to 64, bf16
# (0.64 and 1.0 GB: the runtime's own memory, its scratch above all, comes and
# goes by some 0.15 GB)
@pytest.mark.parametrize("H,M,B,dense", [(120, 10, 4096, True), (60, 64, 2048, False)])
def test_spike_matrices(H, M, B, dense):
    gsbn_amd.release_memory()
    ring = 128 * B * ((H * M + 63) // 64 * 64)
    with_handle, (rc, args) = _taken(lambda: _handle(H, M, B))
    assert (with_handle > ring // 2) == dense
    assert _taken(lambda: rc.run(*args, 0, time_support=True))[0] < ring // 2
    assert _taken(lambda: rc.run(*args, 3))[0] < ring // 2
    timed, out = _taken(lambda: rc.run(*args, 3, time_support=True))
    assert (timed > ring // 2) != dense
    assert out[3] > 0
    rc.close()
