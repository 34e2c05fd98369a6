"""Scratch memory: what a call takes beyond its operands and results is bounded,
and where there is less room (MGW_ALLOC_LIMIT caps a context's bytes) the call
runs with less of it instead of being refused."""
import numpy as np
import pytest

from molgw_amd.gw import Engine, selfenergy_set_state_range
from molgw_amd.workloads import dense_ri, synthetic_system
from oracle import gw_oracle as O

pytestmark = pytest.mark.gpu
MIB = 1 << 20


def loaded(s):
    eng = Engine(0)
    eng.set_eri_3center(s.eri_3center, s.index_basis, s.nbf)
    eng.set_mo(s.c_matrix, s.energy, s.occupation)
    return eng


# K splits of 63 MiB (more than the factorisation's work matrix, which comes
# after it) and of 32 MiB (less)
@pytest.mark.parametrize('nbf, naux, nocc, nomega', [(96, 336, 20, 32), (180, 1000, 80, 16), (150, 700, 50, 32)])
def test_chi0_k_split_workspace(monkeypatch, nbf, naux, nocc, nomega):
    s = synthetic_system(nbf, naux, nocc, seed=23, scale=0.3)
    npole = nocc * (nbf - nocc)
    rng = selfenergy_set_state_range(s.occupation)
    om, wt = np.linspace(0.1, 3.0, nomega), np.linspace(1.0, 0.2, nomega)
    with loaded(s) as eng:
        before = eng.memory()[0]
        ref = eng.polarizability_grid(rng, om, wt)
        held = eng.memory()[0]
    # half transform, (P|ia) and its block, weights, 1 - chi0 and as much for the factorisation
    operands = 8 * (naux * nbf * nocc + 2 * naux * npole + npole * nomega + 2 * naux * naux * nomega)
    assert held - before <= operands + 129 * MIB
    with loaded(s) as eng:
        limit = held - 24 * MIB
        monkeypatch.setenv('MGW_ALLOC_LIMIT', str(limit))
        for _ in range(2):
            got = eng.polarizability_grid(rng, om, wt)
            assert eng.memory()[0] <= limit
            np.testing.assert_allclose(got[:2], ref[:2], rtol=1e-11)


def test_exchange_k_split_workspace(monkeypatch):
    s = synthetic_system(202, 560, 33, seed=24, scale=0.3)
    x = s.c_matrix[:, :33]
    with loaded(s) as eng:
        ref = eng.hartree_exchange_ri(x)
        held = eng.memory()[0]
    with loaded(s) as eng:
        limit = held - 8 * MIB
        monkeypatch.setenv('MGW_ALLOC_LIMIT', str(limit))
        for _ in range(2):
            got = eng.hartree_exchange_ri(x)
            assert eng.memory()[0] <= limit
            for a, b in zip(got, ref):
                np.testing.assert_allclose(a, b, rtol=0, atol=1e-11 * np.max(np.abs(b)))


def test_column_dot_partials(monkeypatch):
    """The FP64 W.B product's partial dots: no more than 256 MiB or what 128-row
    blocks take, and a frequency at a time where there is less room; the same
    result bit for bit."""
    nbf, naux, nomega = 250, 256, 512
    s = synthetic_system(nbf, naux, 3, seed=25, scale=0.3)
    rng = selfenergy_set_state_range(s.occupation)
    om, wt = np.linspace(0.1, 3.0, nomega), np.ones(nomega)
    wc = 0.05j * np.arange(3) - 0.1
    cols = nbf * nbf
    with loaded(s) as eng:
        eng.polarizability_grid(rng, om, wt)
        before = eng.memory()[0]
        ref = eng.gw_selfenergy_imag(rng, wc)
        held = eng.memory()[0]
    # (P|pm), the half transform, the dots and their partials
    operands = 8 * (naux * cols + naux * nbf * nbf + cols * nomega)
    assert held - before <= operands + 8 * 2 * cols * nomega + MIB
    with loaded(s) as eng:
        eng.polarizability_grid(rng, om, wt)
        limit = eng.memory()[0] + operands + 16 * MIB
        monkeypatch.setenv('MGW_ALLOC_LIMIT', str(limit))
        got = eng.gw_selfenergy_imag(rng, wc)
        assert eng.memory()[0] <= limit
    np.testing.assert_array_equal(got, ref)


def test_contour_dot_partials(monkeypatch):
    s = synthetic_system(60, 200, 8, seed=26, scale=0.3)
    rng = selfenergy_set_state_range(s.occupation)
    omega = np.linspace(-0.1, 0.1, 5)
    e0 = s.energy[rng.nsemin - 1:rng.nsemax]
    with loaded(s) as eng:
        ref, _ = eng.gw_selfenergy_contour(rng, omega, e0, 12)
        held = eng.memory()[0]
    with loaded(s) as eng:
        # 14 frequencies, 4 row blocks: 1.5 MiB of partial dots
        limit = held - MIB
        monkeypatch.setenv('MGW_ALLOC_LIMIT', str(limit))
        got, _ = eng.gw_selfenergy_contour(rng, omega, e0, 12)
        assert eng.memory()[0] <= limit
    np.testing.assert_array_equal(got, ref)


def test_qs_state_products(monkeypatch):
    """The QS self-energy's products of the single states i: 1 GiB of them at a
    time also where there are fewer poles than states, and fewer where there is
    less room."""
    n, naux = 640, 4
    s = synthetic_system(n, naux, 5, seed=27, scale=0.3)
    g = np.random.default_rng(28)
    pole, ws = np.array([0.4, 1.1]), g.standard_normal((naux, 2))
    rng = selfenergy_set_state_range(s.occupation)
    with loaded(s) as eng:
        eng.set_spectral_function(pole, ws)
        before = eng.memory()[0]
        ref, _ = eng.gw_selfenergy_qs(rng, eta=0.05)
        held = eng.memory()[0]
    # (P|pi) and its half transform, w and its scaled copy, the result
    operands = 8 * (2 * naux * n * n + 2 * 2 * n * n + 4 * n * n)
    assert held - before <= operands + 1024 * MIB + MIB
    epi = np.einsum('pkl,km,li->pmi', dense_ri(s), s.c_matrix, s.c_matrix, optimize=True)
    want = O.gw_selfenergy_qs(epi, ws, pole, s.energy, s.occupation, rng, eta=0.05)
    # each entry: 2 n terms of at most max w^2 / eta, each off by a few times naux 2^-53
    w = np.einsum('ps,pmi->smi', ws, epi)
    size = np.einsum('smi->m', w * w) / 0.05
    bound = 4 * (2 * naux + 2 * n) * 2.0 ** -53 * np.sqrt(size[:, None] * size[None, :])
    assert np.all(np.abs(ref - want) <= bound)
    for room in (64 * MIB, MIB):
        with loaded(s) as eng:
            eng.set_spectral_function(pole, ws)
            limit = eng.memory()[0] + operands + room
            monkeypatch.setenv('MGW_ALLOC_LIMIT', str(limit))
            got, _ = eng.gw_selfenergy_qs(rng, eta=0.05)
            monkeypatch.delenv('MGW_ALLOC_LIMIT')
            assert eng.memory()[0] <= limit
            assert np.all(np.abs(got - want) <= bound)


def test_pole_self_energy_partial_sums():
    """256 MiB of partial sums however many poles and frequencies there are; the
    frequencies of one launch do not change another's result."""
    n, naux, npole = 60, 2, 1000000
    s = synthetic_system(n, naux, 5, seed=29, scale=0.3)
    g = np.random.default_rng(30)
    pole, ws = np.sort(g.uniform(0.4, 3.0, npole)), g.standard_normal((naux, npole)) * 1e-3
    rng = selfenergy_set_state_range(s.occupation)
    omega = np.linspace(-0.3, 0.3, 300)
    with loaded(s) as eng:
        eng.set_spectral_function(pole, ws)
        before = eng.memory()[0]
        got, egw = eng.gw_selfenergy(rng, omega, s.energy, eta=0.05)
        held = eng.memory()[0]
        sub, sub_egw = eng.gw_selfenergy(rng, omega[100:104], s.energy, eta=0.05)
    # w of two states i, the half transform and (P|pi), the result
    operands = 8 * (2 * npole * n + 2 * naux * n * n + 2 * 300 * n)
    assert held - before <= operands + 257 * MIB
    # the poles' sums are taken in another order: npole n terms of one sign each
    scale = np.max(np.abs(got))
    assert np.max(np.abs(sub - got[100:104])) <= 2 * npole * n * 2.0 ** -53 * scale and abs(sub_egw - egw) <= 1e-9 * abs(egw)
