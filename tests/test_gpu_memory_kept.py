"""Device memory that a closed solver leaves (-m gpu): it is kept, it serves an
equal solver without more from the device, and two solvers open at once have
memory of their own."""

import gc
import time

import pytest
import torch

import gsbn_amd
import oracle as O
from gsbn_amd import Solver, configs
from helpers import compare_state

pytestmark = pytest.mark.gpu

# bytes of the network's synapse records, 0.86 GB (the runtime's own memory, its
# scratch above all, comes and goes by some 0.15 GB)
SYNAPSES = 100 * 99 * 60 * 60 * 24


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


def _open(spec, path):
    path.mkdir(exist_ok=True)
    s = Solver(configs.write(spec, str(path)))
    configs.apply_conn_arrays(s, spec)
    return s


def test_kept_and_used_again(tmp_path):
    spec = configs.recall_net(100, 60, 2, 60, 5, 30, 0.5, name="big")
    gsbn_amd.release_memory()
    before = _free()
    s = _open(spec, tmp_path)
    s.step(90)
    s.close()
    kept = before - _free()
    assert SYNAPSES // 2 < kept <= torch.cuda.mem_get_info()[1] // 8
    s = _open(spec, tmp_path)
    s.step(90)
    assert before - _free() < kept + SYNAPSES // 2
    s.close()
    gsbn_amd.release_memory()
    assert before - _free() < SYNAPSES // 2


def test_two_open_at_once(tmp_path):
    """The second's arrays come from memory that earlier solvers left, while the
    first is open and goes on being read."""
    big = configs.recall_net(30, 40, 2, 60, 5, 30, 0.5, name="big")
    _open(big, tmp_path / "x").close()
    a = _open(configs.recall_net(9, 11, 2, 40, 5, 20, 0.5, seed=1, reset=6, name="a"), tmp_path / "a")
    a.step(90)
    names = ("wij_0", "pij_0", "tij_0", "pj_0", "spike_0", "epsc_0")
    want = {n: a.vector(n) for n in names}
    spec = configs.recall_net(12, 9, 2, 40, 5, 20, 0.5, seed=2, reset=6, name="b")
    b = _open(spec, tmp_path / "b")
    ora = O.OracleNet(spec)
    for _ in range(90):
        b.step(1)
        ora.step()
    assert not compare_state(b, ora, spec)
    for n in names:
        assert a.vector(n).tobytes() == want[n].tobytes(), n
    a.close()
    assert not compare_state(b, ora, spec)
    b.close()
