"""The AO->MO transform's column tiles of 16 FN columns: windows at and beside
the tiles' edges for every FN that the rule picks. Bound: a sum of K products
in any order is off by at most K 2^-53 sum |a b|, here K = nbf twice, and twice
that for the two sides' roundings."""
import numpy as np
import pytest

from molgw_amd.gw import Engine
from molgw_amd.workloads import dense_ri, synthetic_system

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -53
NBF, NAUX = 177, 259       # 3 row tiles x 177 products: past the 512 workgroups that the column tiles ask for


def column_tile(n, k):
    """The rule of narrow_fn (gemm_f64.hip); 0 for the 128-wide tiles."""
    weight = {1: 1 / 23, 2: 2 / 38, 3: 3 / 42, 4: 4 / 48, 5: 5 / 58, 6: 6 / 53, 8: 8 / 65}
    cost = {fn: -(-n // (16 * fn)) * w * (k + (150 if fn == 8 else 60)) for fn, w in weight.items()}
    best = min(sorted(cost, reverse=True), key=lambda fn: cost[fn])
    return 0 if best == 8 else best


@pytest.fixture(scope='module')
def loaded():
    s = synthetic_system(NBF, NAUX, 9, seed=22, scale=0.3)
    with Engine(0) as e:
        e.set_eri_3center(s.eri_3center, s.index_basis, s.nbf)
        e.set_mo(s.c_matrix, s.energy, s.occupation)
        yield e, s, dense_ri(s)


@pytest.mark.parametrize('ncol, fn', [(1, 1), (15, 1), (16, 1), (17, 2), (31, 2), (32, 2), (33, 3), (47, 3), (48, 3),
                                      (49, 4), (64, 4), (65, 5), (79, 5), (80, 5), (81, 6), (95, 6), (96, 6), (97, 4),
                                      (112, 4), (129, 5), (161, 6), (176, 6)])
def test_every_column_tile(loaded, ncol, fn):
    eng, s, b = loaded
    assert column_tile(ncol, NBF) == fn and -(-NAUX // 128) * -(-ncol // 112) * NBF >= 512
    eng.destroy_eri_3center_mo()
    got = eng.calculate_eri_3center_mo(1, s.nstate, 2, ncol + 1)
    eng.destroy_eri_3center_mo()
    c = s.c_matrix
    ref = np.einsum('pkn,km->pmn', b @ c[:, 1:ncol + 1], c, optimize=True)
    size = np.einsum('pkn,km->pmn', np.abs(b) @ np.abs(c[:, 1:ncol + 1]), np.abs(c), optimize=True)
    assert np.all(np.abs(got - ref) <= 4 * s.nbf * EPS * size)


def test_no_shape_takes_a_seventh_tile():
    """112 columns cost more than 128 (a column at 56 against 65 TFLOP/s), so
    the tiles end at 96."""
    assert {column_tile(n, k) for n in range(1, 1024) for k in (16, 60, 177, 1000, 10 ** 5)} == set(range(7))
