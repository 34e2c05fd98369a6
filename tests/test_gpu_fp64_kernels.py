"""FP64 kernels at the sizes where their tiles, splits and remainders change:
the MFMA GEMM's column tiles and K splits, the Hartree/exchange build, the
pole self-energy's frequency groups and the QS self-energy's batched sum.

Bounds: a sum of K products in any order is off by at most K 2^-53 sum |a b|
(K here the longest chain of products), so each test forms sum |a b| in numpy
and allows twice that bound, for the two sides' roundings."""
import numpy as np
import pytest

from molgw_amd.gw import Engine, selfenergy_set_state_range
from molgw_amd.workloads import dense_ri, synthetic_system
from oracle import gw_oracle as O

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -53


@pytest.fixture(scope='module')
def eng():
    with Engine(0) as e:
        yield e


def _load(eng, s):
    eng.set_eri_3center(s.eri_3center, s.index_basis, s.nbf)
    eng.set_mo(s.c_matrix, s.energy, s.occupation)


@pytest.mark.parametrize('ncol', [1, 15, 16, 17, 33, 49, 64, 65, 80, 81, 97, 112, 113, 128])
def test_ao2mo_column_tiles(eng, ncol):
    """(P|m n) for windows that fall on and beside the column tiles."""
    s = synthetic_system(131, 259, 9, seed=11, scale=0.3)
    _load(eng, s)
    eng.destroy_eri_3center_mo()
    got = eng.calculate_eri_3center_mo(1, s.nstate, 2, ncol + 1)
    eng.destroy_eri_3center_mo()
    b, c = dense_ri(s), s.c_matrix
    ref = np.einsum('pkn,km->pmn', b @ c[:, 1:ncol + 1], c, optimize=True)
    size = np.einsum('pkn,km->pmn', np.abs(b) @ np.abs(c[:, 1:ncol + 1]), np.abs(c), optimize=True)
    assert np.all(np.abs(got - ref) <= 4 * s.nbf * EPS * size)


@pytest.mark.parametrize('nbf, naux, nocc, nomega', [(24, 65, 5, 1), (70, 63, 20, 1), (90, 129, 30, 2), (131, 192, 40, 3)])
def test_chi_with_split_transitions(eng, nbf, naux, nocc, nomega):
    """chi(i omega) where few tiles and many transitions split the K range;
    chi = (1 - chi0)^-1 - 1 with |(1 - chi0)^-1| <= 1, so its error is that of
    chi0 and of the factorisation's n products."""
    s = synthetic_system(nbf, naux, nocc, seed=12, scale=0.3)
    _load(eng, s)
    om = np.linspace(0.3, 2.0, nomega)
    _, _, chi = eng.polarizability_grid(selfenergy_set_state_range(s.occupation), om, np.ones(nomega), return_chi=True)
    b, c = dense_ri(s), s.c_matrix
    x = np.einsum('pkl,ka,li->pia', b, c[:, nocc:], c[:, :nocc], optimize=True).reshape(naux, -1)
    de = (s.energy[None, nocc:] - s.energy[:nocc, None]).reshape(-1)
    for f in range(nomega):
        w = 4.0 * de / (om[f] ** 2 + de ** 2)
        chi0 = (x * w) @ x.T
        ref = np.linalg.inv(np.eye(naux) + chi0) - np.eye(naux)
        bound = 4 * (len(de) + naux) * EPS * (1.0 + np.trace(chi0))
        assert np.max(np.abs(chi[:, :, f] - ref)) <= bound


@pytest.mark.parametrize('nbf, naux, nx', [(1, 1, 1), (2, 3, 1), (7, 5, 3), (24, 84, 5), (33, 130, 33), (65, 64, 2),
                                           (130, 257, 17), (131, 300, 81)])
def test_hartree_exchange(eng, nbf, naux, nx):
    s = synthetic_system(nbf, naux, 1, seed=13, scale=0.3)
    eng.set_eri_3center(s.eri_3center, s.index_basis, s.nbf)
    x = np.random.default_rng(14).standard_normal((nbf, nx))
    j, k = eng.hartree_exchange_ri(x, spin_fact=2.0)
    b = dense_ri(s)
    h, ha = b @ x, np.abs(b) @ np.abs(x)
    jref = np.einsum('pkl,p->kl', b, 2.0 * np.einsum('pki,ki->p', h, x))
    jsize = np.einsum('pkl,p->kl', np.abs(b), 2.0 * np.einsum('pki,ki->p', ha, np.abs(x)))
    kref = -np.einsum('pki,pli->kl', h, h, optimize=True)
    ksize = np.einsum('pki,pli->kl', ha, ha, optimize=True)
    chain = nbf + nbf * nx + naux * max(1, nx)
    assert np.all(np.abs(j - jref) <= 2 * chain * EPS * jsize)
    assert np.all(np.abs(k - kref) <= 2 * chain * EPS * ksize)
    np.testing.assert_array_equal(j, j.T)
    np.testing.assert_array_equal(k, k.T)


@pytest.mark.parametrize('nomega', [1, 3, 4, 5, 51, 63, 64, 65, 254, 255, 256, 300])
def test_pole_self_energy_frequency_groups(eng, nomega):
    """Sigma(omega) for frequency counts on both sides of the thread groups and
    launches, on more than one block of poles; no frequency lies within eta of
    a pole by construction, so a term's relative error is a few roundings."""
    s = synthetic_system(40, 60, 15, seed=15, scale=0.3)       # 375 transitions
    t = synthetic_system(60, 60, 14, seed=16, scale=0.3)       # 644: two blocks of poles
    for sys in (s, t):
        _load(eng, sys)
        rng = selfenergy_set_state_range(sys.occupation, selfenergy_state_min=sys.nocc - 1,
                                         selfenergy_state_max=sys.nocc + 2)
        _, _, pole, ws = eng.polarizability(rng, return_ws=True)
        omega = np.linspace(-0.2, 0.2, nomega) if nomega > 1 else np.zeros(1)
        e0 = sys.energy[rng.nsemin - 1:rng.nsemax]
        got, egw = eng.gw_selfenergy(rng, omega, e0, eta=0.05)
        b, c = dense_ri(sys), sys.c_matrix
        mo = np.einsum('pkl,km,ln->pmn', b, c[:, rng.nsemin - 1:rng.nsemax], c, optimize=True)
        ref_egw = 0.0
        for m in range(rng.nse):
            w2 = (ws.T @ mo[:, m, :]) ** 2
            x = (e0[m] + omega)[:, None, None] - sys.energy[None, None, :]
            occ = (np.arange(sys.nstate) < sys.nocc)[None, None, :]
            d = np.where(occ, x + pole[None, :, None] - 0.05j, x - pole[None, :, None] + 0.05j)
            ref = (w2[None] / d).sum((1, 2))
            size = (w2[None] / np.abs(d)).sum((1, 2))
            # w = ws^T (P|pi) carries naux products, its square twice that, the sum npole nstate terms
            assert np.all(np.abs(got[:, m] - ref) <= (4 * 60 + 2 * len(pole) * sys.nstate) * EPS * size * 20)
            if m + rng.nsemin <= sys.nocc:
                ref_egw += 2.0 * np.sum(w2[:, sys.nocc:] / (e0[m] - sys.energy[None, sys.nocc:] - pole[:, None]))
        assert abs(egw - ref_egw) <= 1e-10 * max(1.0, abs(ref_egw))


@pytest.mark.parametrize('lo, hi, ncore', [(1, 30, 0), (5, 5, 0), (3, 9, 2), (1, 17, 0)])
def test_qs_self_energy_batched_sum(eng, lo, hi, ncore):
    s = synthetic_system(30, 70, 8, seed=17, scale=0.3)
    _load(eng, s)
    rng = selfenergy_set_state_range(s.occupation, ncoreg=ncore, selfenergy_state_min=lo, selfenergy_state_max=hi)
    _, _, pole, ws = eng.polarizability(rng, return_ws=True)
    mo, _ = eng.gw_selfenergy_qs(rng, eta=0.05)
    b, c = dense_ri(s), s.c_matrix
    win = slice(rng.nsemin - 1, rng.nsemax)
    epi = np.einsum('pkl,km,li->pmi', b, c[:, win], c[:, ncore:rng.nvirtual_G - 1], optimize=True)
    ref = O.gw_selfenergy_qs(epi, ws, pole, s.energy, s.occupation, rng, eta=0.05)
    size = sum((np.abs(ws.T @ epi[:, :, k]).T @ np.abs(ws.T @ epi[:, :, k])) / 0.05 for k in range(epi.shape[2]))
    assert np.all(np.abs(mo[win, win] - ref) <= 4 * (70 + len(pole) * epi.shape[2]) * EPS * size)


@pytest.mark.parametrize('naux', [1, 2, 15, 16, 17, 33, 63, 64, 65, 112, 113, 127, 128, 129, 145])
def test_chi_leaf_sizes(eng, naux):
    """(1 - chi0)^-1 of sizes on both sides of the factorisation's blocks of 16
    and leaves of 64 and 128; bound as in test_chi_with_split_transitions."""
    s = synthetic_system(20, naux, 6, seed=19, scale=0.3)
    _load(eng, s)
    om = np.array([0.2, 1.0, 5.0])
    _, _, chi = eng.polarizability_grid(selfenergy_set_state_range(s.occupation), om, np.ones(3), return_chi=True)
    b, c = dense_ri(s), s.c_matrix
    x = np.einsum('pkl,ka,li->pia', b, c[:, 6:], c[:, :6], optimize=True).reshape(naux, -1)
    de = (s.energy[None, 6:] - s.energy[:6, None]).reshape(-1)
    for f in range(3):
        chi0 = (x * (4.0 * de / (om[f] ** 2 + de ** 2))) @ x.T
        ref = np.linalg.inv(np.eye(naux) + chi0) - np.eye(naux)
        assert np.max(np.abs(chi[:, :, f] - ref)) <= 4 * (len(de) + naux) * EPS * (1.0 + np.trace(chi0))
