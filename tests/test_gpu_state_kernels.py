"""The kernels that end an imaginary-axis solve, at the edges of how they divide
their work: the sum over (state, frequency) terms, whose spare threads take
further frequencies up to 128 states, and the graphical QP solution on a wave
per state (64 intervals of the frequency grid at a time, up to four roots kept).
Bounds: the sum's terms are each correct to a few 2^-53, so two orders differ by
at most (count + 16) 2^-53 of the sum of their sizes; the QP roots come from the
same expressions as the reference's but for the order of f = sigma + exc + e0, whose
few 2^-53 |f| a slope between points h apart carries to the weight z = 1 / (1 -
slope) times z^2 / h, and to the root times z."""
import numpy as np
import pytest

from molgw_amd.gw import Engine, selfenergy_set_state_range
from molgw_amd.workloads import synthetic_system
from oracle import gw_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('nbf, nomega', [(3, 1), (5, 60), (64, 5), (85, 4), (127, 3), (128, 9), (129, 7), (130, 17)])
def test_imaginary_sum(nbf, nomega):
    s = synthetic_system(nbf, 20, 2, seed=nbf, scale=0.3)
    om, wt = np.linspace(0.1, 4.0, nomega), np.linspace(0.5, 1.5, nomega)
    wc = 0.05 + 0.3j * np.arange(4)
    with Engine(0) as e:
        e.set_eri_3center(s.eri_3center, s.index_basis, nbf)
        e.set_mo(s.c_matrix, s.energy, s.occupation)
        rng = selfenergy_set_state_range(s.occupation, selfenergy_state_range=1)
        _, _, chi = e.polarizability_grid(rng, om, wt, return_chi=True)
        got = e.gw_selfenergy_imag(rng, wc)
        b = e.calculate_eri_3center_mo(1, nbf, rng.nsemin, rng.nsemax)       # (P, p, m)
    v = np.einsum('Ppm,PQk,Qpm->pmk', b, chi, b, optimize=True)
    va = np.einsum('Ppm,PQk,Qpm->pmk', np.abs(b), np.abs(chi), np.abs(b), optimize=True)
    z = wc[:, None, None] - s.energy[None, :, None]
    g = -wt / (2 * np.pi) * (1 / (z + 1j * om) + 1 / (z - 1j * om))          # (kc, p, k)
    ref = np.einsum('cpk,pmk->cm', g, v)
    size = np.einsum('cpk,pmk->cm', np.abs(g), va)
    chain = nbf * nomega + 2 * 20 * 20 + 20 ** 2 + 64                         # sums, products, factorisation
    assert np.all(np.abs(got - ref) <= 4 * chain * 2.0 ** -53 * size)


@pytest.mark.parametrize('nomega', [1, 3, 63, 65, 67, 129, 201])
def test_graphical_solution(nomega):
    n = 9
    r = np.random.default_rng(nomega)
    s = synthetic_system(n, 12, 3, seed=1, scale=0.3)
    omega = 0.005 * (np.arange(nomega) - nomega // 2)
    with Engine(0) as e:
        e.set_eri_3center(s.eri_3center, s.index_basis, n)
        e.set_mo(s.c_matrix, s.energy, s.occupation)
        rng = selfenergy_set_state_range(s.occupation)
        nse = rng.nse
        # up to a dozen crossings a state, some of them with the same weight
        wave = np.sin(np.arange(nse)[None, :] * omega[:, None] * 60.0) * 0.05 + 0.01 * r.standard_normal((nomega, nse))
        sigma = wave + 0.5 * omega[:, None] + 0j
        e0 = s.energy
        se0, exc = e0[rng.nsemin - 1:rng.nsemax], 0.002 * r.standard_normal(n)
        eqp, zz, _ = e.find_qp_energy(rng, omega, sigma, se0, exc, e0)
    want, wz = O.find_qp_energy_graphical(sigma, omega, se0, exc, e0, O.selfenergy_set_state_range(s.occupation[:, None]))
    eps = 16 * 2.0 ** -53 * (1.0 + np.max(np.abs(sigma)) + np.max(np.abs(e0)) + np.max(np.abs(omega)))
    assert np.all(np.abs(zz - wz) <= eps * (1.0 + wz ** 2 / 0.005))
    assert np.all(np.abs(eqp - want) <= eps * (1.0 + wz))
