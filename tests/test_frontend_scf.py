"""The RI-HF iteration far from convergence, and what it says when it stops
early (CPU)."""
import os
import warnings

import numpy as np
import pytest

from molgw_amd.frontend import alkane, run_rihf, water_cluster
from molgw_amd.frontend.scf import _NextFock
from tests.conftest import GOLDEN

BASIS = os.path.join(GOLDEN, 'basis')


def test_early_end_is_told():
    mol = water_cluster(1)
    with pytest.warns(UserWarning, match='not converged in 3 iterations'):
        r = run_rihf(mol, 'cc-pVDZ', 'cc-pVDZ-RI', BASIS, max_iter=3)
    assert not r.converged and r.iterations == 3
    with warnings.catch_warnings():
        warnings.simplefilter('error')
        r = run_rihf(mol, 'cc-pVDZ', 'cc-pVDZ-RI', BASIS)
    assert r.converged


@pytest.mark.parametrize('diis', [0, 1, 2, 8])
def test_methane_for_every_history_length(diis):
    ref = run_rihf(alkane(1), 'cc-pVDZ', 'cc-pVDZ-RI', BASIS)
    r = run_rihf(alkane(1), 'cc-pVDZ', 'cc-pVDZ-RI', BASIS, diis=diis)
    assert r.converged and abs(r.energy - ref.energy) < 1e-9


def test_damped_steps_never_raise_the_energy():
    """On a model quadratic in the density, E(D) = tr h D + tr D G(D) / 2 with a
    symmetric positive G, from a start without a gap."""
    g = np.random.default_rng(0)
    n, nocc = 24, 7
    h = 0.05 * g.standard_normal((n, n))
    h = h + h.T
    a = g.standard_normal((60, n, n))
    a = 0.3 * (a + a.transpose(0, 2, 1))

    def fock(d):
        return h + np.einsum('pij,p->ij', a, np.einsum('pkl,kl->p', a, d))

    step = _NextFock(8)
    c = np.linalg.eigh(h)[1]
    energies = []
    for _ in range(12):
        d = 2.0 * c[:, :nocc] @ c[:, :nocc].T
        f = fock(d)
        if np.abs(f @ d - d @ f).max() < step.FAR:
            break
        used = step(d, f, f @ d - d @ f)
        dm, fm = step.mixed
        assert used is fm
        np.testing.assert_allclose(fm, fock(dm), atol=1e-9)      # the mixed Fock matrix is that of the mixed density
        energies.append(0.5 * np.sum(dm * (h + fm)))
        c = np.linalg.eigh(used)[1]
    assert len(energies) > 3 and all(b <= a + 1e-12 * abs(a) for a, b in zip(energies, energies[1:]))
