"""Scratch memory: what a call takes beyond its operands and results is bounded,
and where there is less room (MGW_ALLOC_LIMIT caps a context's bytes) the call
runs with less of it instead of being refused."""
import numpy as np
import pytest

from molgw_amd.gw import Engine, selfenergy_set_state_range
from molgw_amd.workloads import synthetic_system

pytestmark = pytest.mark.gpu
MIB = 1 << 20


def loaded(s):
    eng = Engine(0)
    eng.set_eri_3center(s.eri_3center, s.index_basis, s.nbf)
    eng.set_mo(s.c_matrix, s.energy, s.occupation)
    return eng


# K splits of 64 MiB (more than the factorisation's work matrix, which comes
# after it) and of 32 MiB (less)
@pytest.mark.parametrize('nbf, naux, nocc, nomega', [(180, 1000, 80, 16), (150, 700, 50, 32)])
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
