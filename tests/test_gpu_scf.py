"""RI-HF of long alkanes on the GPU: their core-Hamiltonian guess has no gap, and
the iteration has to come out of it whatever the last bits of the integrals are.
C18H38: the energy of the host route (host integrals, numpy J and K)."""
import os

import numpy as np
import pytest

from molgw_amd.frontend import alkane, run_rihf_device
from molgw_amd.gw import Engine
from tests.conftest import GOLDEN

pytestmark = pytest.mark.gpu
BASIS = os.path.join(GOLDEN, 'basis')


@pytest.mark.parametrize('n', [13, 18, 24])
def test_long_alkanes_converge(n):
    with Engine(0) as eng:
        r = run_rihf_device(alkane(n), 'cc-pVDZ', 'cc-pVDZ-RI', BASIS, eng)
    if n == 18:
        assert abs(r.energy + 703.8280676) < 1e-6
    assert r.energy_mo[r.nocc] - r.energy_mo[r.nocc - 1] > 0.5
    # the Fock matrix commutes with its density
    fds = r.hamiltonian_fock @ (r.c_matrix[:, :r.nocc] @ r.c_matrix[:, :r.nocc].T) @ r.s_matrix
    assert np.max(np.abs(fds - fds.T)) < 1e-5
    assert r.converged and r.iterations <= 40
