"""Device memory from one solver to the next (-m gpu): a solver on memory that
another left behind runs as on fresh memory, and the memory can be given back."""

import pytest
import torch

import gsbn_amd
import oracle as O
from gsbn_amd import Solver, configs
from helpers import compare_state

pytestmark = pytest.mark.gpu


def _run(spec, path):
    path.mkdir(exist_ok=True)
    s = Solver(configs.write(spec, str(path)))
    configs.apply_conn_arrays(s, spec)
    s.step(90)
    return s


def test_a_solver_on_left_memory(tmp_path):
    big = configs.recall_net(40, 50, 2, 60, 5, 30, 0.5, name="big")
    for i, prec in enumerate(("fp32", "fp16", "fp32")):
        big.trace_precision = prec
        _run(big, tmp_path / ("b%d" % i)).close()
        spec = configs.recall_net(9, 11, 2, 40, 5, 20, 0.5, seed=i, reset=6, name="small")
        s = _run(spec, tmp_path / ("s%d" % i))
        ora = O.OracleNet(spec)
        for _ in range(90):
            ora.step()
        assert not compare_state(s, ora, spec)
        s.close()


def test_left_memory_is_given_back(tmp_path):
    spec = configs.recall_net(60, 60, 2, 60, 5, 30, 0.5, name="big")  # 0.6 GB
    gsbn_amd.release_memory()
    before = torch.cuda.mem_get_info()[0]
    _run(spec, tmp_path).close()
    kept = before - torch.cuda.mem_get_info()[0]
    assert 0 <= kept <= torch.cuda.mem_get_info()[1] // 8
    gsbn_amd.release_memory()
    assert before - torch.cuda.mem_get_info()[0] < (64 << 20)
