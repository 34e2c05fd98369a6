"""HIP-graph replay of the batched Cholesky sequence when a switch that decides
its kernels changes between two solves of the same buffers."""
import numpy as np
import pytest

from molgw_amd.gw import Engine
from molgw_amd.workloads import synthetic_system
from tests.test_gpu_graphs import grid_solve

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('precision', ['fp64', 'fp16x3'])
def test_replay_follows_the_leaf_choice(monkeypatch, precision):
    """MGW_CHOL_LEAF is read at every factorisation, replayed ones included."""
    s = synthetic_system(70, 300, 11, seed=51, scale=0.3)
    ref = {}
    with Engine(0) as eager:
        for leaf in ('1', '0'):
            monkeypatch.setenv('MGW_CHOL_LEAF', leaf)
            ref[leaf] = grid_solve(eager, s, precision)
    assert np.any(ref['0'][2] != ref['1'][2])
    with Engine(0) as eng:
        eng.graphs(True)
        for leaf in ('1', '0', '1', '0', '0', '1'):
            monkeypatch.setenv('MGW_CHOL_LEAF', leaf)
            got = grid_solve(eng, s, precision)
            assert got[:2] == ref[leaf][:2]
            np.testing.assert_array_equal(got[2], ref[leaf][2])
