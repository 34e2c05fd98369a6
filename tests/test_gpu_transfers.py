"""Vectors on their way to and from the device: sizes around the half of the
128 KiB of pinned memory up to which they are staged, more of them in one call
than it holds, host arrays written again right after the call that read them,
and the transition table of fractional occupations."""
import numpy as np
import pytest

from molgw_amd.gw import Engine, StateRanges
from molgw_amd.workloads import dense_ri, synthetic_system

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -53


@pytest.mark.parametrize('nbf', [3, 89, 90, 91, 128, 131])
def test_transfers_around_the_staged_size(nbf):
    # nbf^2 doubles: 64 800 bytes at 90, 66 248 at 91; 128^2 doubles fill the memory
    s = synthetic_system(nbf, 40, 2, seed=nbf, scale=0.3)
    b = dense_ri(s)
    with Engine(0) as e:
        e.set_eri_3center(s.eri_3center, s.index_basis, nbf)
        c, energy, occ = np.asfortranarray(s.c_matrix).copy(order='F'), s.energy.copy(), s.occupation.copy()
        e.set_mo(c, energy, occ)
        c[:], energy[:], occ[:] = np.nan, np.nan, np.nan
        got = e.calculate_eri_3center_mo(1, nbf, 1, 2)
        cs = s.c_matrix
        ref = np.einsum('pkn,km->pmn', b @ cs[:, :2], cs, optimize=True)
        size = np.einsum('pkn,km->pmn', np.abs(b) @ np.abs(cs[:, :2]), np.abs(cs), optimize=True)
        assert np.all(np.abs(got - ref) <= 4 * nbf * EPS * size)
        for nx in (1, nbf):
            x = cs[:, :nx]
            j, k = e.hartree_exchange_ri(x, spin_fact=2.0)
            h = b @ x
            kr = -np.einsum('pai,pbi->ab', h, h, optimize=True)
            ks = np.einsum('pai,pbi->ab', np.abs(b) @ np.abs(x), np.abs(b) @ np.abs(x), optimize=True)
            assert np.all(np.abs(k - kr) <= 4 * (nbf + 40 * nx) * EPS * ks)


@pytest.mark.parametrize('nspin, ncore, nvirtual', [(1, 0, 31), (1, 3, 25), (2, 0, 31), (2, 5, 12), (1, 29, 31)])
def test_transition_count_of_any_occupations(nspin, ncore, nvirtual):
    n, fact = 30, 2.0          # the full occupation that the count assumes
    s = synthetic_system(n, 12, 5, seed=4, scale=0.3)
    rng = np.random.default_rng(ncore + nspin)
    occ = rng.choice([0.0, 1e-6, 2e-5, 0.3, 0.3, fact / 2, fact - 2e-5, fact - 1e-6, fact], size=(n, nspin))
    want = 0
    for q in range(nspin):
        for i in range(max(ncore, 0), min(n, nvirtual - 1)):
            for j in range(max(ncore, 0), min(n, nvirtual - 1)):
                oi, oj = occ[i, q], occ[j, q]
                empty, full = oi < 1e-5 and oj < 1e-5, oi > fact - 1e-5 and oj > fact - 1e-5
                want += not (empty or full or oj > oi)
    with Engine(0) as e:
        e.set_eri_3center(s.eri_3center, s.index_basis, n)
        e.set_mo(np.repeat(s.c_matrix[:, :, None], nspin, axis=2), np.repeat(s.energy[:, None], nspin, axis=1), occ)
        r = StateRanges(0, n + 1, 5, 6, 1, 1, ncore, nvirtual)
        assert e.npole(r) == want
