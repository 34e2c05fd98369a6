"""The AO->MO transform of windows at and beside the edges of every tile that the
rule for few columns picks. Bound: a sum of K products in any order is off by at
most K 2^-53 sum |a b|, here K = nbf twice, and twice that for the two sides'
roundings."""
import functools

import numpy as np
import pytest

from molgw_amd.gw import Engine
from molgw_amd.workloads import dense_ri, synthetic_system

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -53


def chosen_tile(m, n, k):
    """(rows, columns) of the tile that column_tiles (gemm_f64.hip) picks."""
    tiles = [(128, 128, 2, 70.4, 126), (64, 64, 4, 63.9, 84.8), (128, 16, 4, 43.0, 31.6), (128, 32, 4, 52.7, 43),
             (128, 48, 4, 65.7, 78.9), (128, 64, 4, 66.2, 88.7), (128, 80, 3, 68.9, 96.2), (128, 96, 3, 67.0, 95)]

    def cost(tile):
        bm, bn, share, rate, fixed = tile
        full, last = divmod(-(-m // bm) * -(-n // bn), 256 * share)
        if bm == 64 and full >= 8:
            return float('inf')
        part = last / (256 * share)
        rounds = 0.33 + 0.67 * part if full == 0 else full + (0.15 + 0.85 * part if last else 0.0)
        return bm * bn * 256 * share / rate * (k + fixed) * rounds
    return min(tiles, key=cost)[:2]


@functools.lru_cache(maxsize=1)
def system(nbf, naux):
    s = synthetic_system(nbf, naux, 9, seed=22, scale=0.3)
    return s, dense_ri(s)


SMALL, LARGE, LARGER, LONG = (131, 129), (177, 371), (309, 637), (400, 196)
WINDOWS = [(*SMALL, n) for n in (1, 15, 16, 17, 31, 33, 64, 65, 130)] + [
    (*LARGE, n) for n in (1, 16, 17, 32, 33, 47, 48, 49, 63, 64, 65, 79, 80, 81, 95, 96, 97, 112, 129, 144, 161, 176)] + [
    (*LARGER, n) for n in (49, 64)] + [(*LONG, n) for n in (85, 95, 96)]


@pytest.mark.parametrize('nbf, naux, ncol', WINDOWS)
def test_windows(nbf, naux, ncol):
    s, b = system(nbf, naux)
    c = s.c_matrix
    with Engine(0) as eng:
        eng.set_eri_3center(s.eri_3center, s.index_basis, s.nbf)
        eng.set_mo(s.c_matrix, s.energy, s.occupation)
        got = eng.calculate_eri_3center_mo(1, s.nstate, 2, ncol + 1)
    if nbf > 300:      # rows of the first and last tiles
        rows = np.r_[0:66, naux - 66:naux]
        b, got = b[rows], got[rows]
    half, size = b @ c[:, 1:ncol + 1], np.abs(b) @ np.abs(c[:, 1:ncol + 1])
    ref = np.einsum('pkn,km->pmn', half, c, optimize=True)
    size = np.einsum('pkn,km->pmn', size, np.abs(c), optimize=True)
    assert np.all(np.abs(got - ref) <= 4 * s.nbf * EPS * size)


def test_windows_reach_every_tile():
    """Of few columns; 128 x 128 is the tile of every larger product."""
    first = {chosen_tile(nbf * naux, n, nbf) for nbf, naux, n in WINDOWS}
    assert first >= {(128, 16 * fn) for fn in range(1, 7)} | {(64, 64)}
    assert chosen_tile(10 ** 6, 128, 2000) == (128, 128)
