"""Three-centre integrals whose ket shells are contracted (an orbital basis in
the auxiliary's place: up to eight primitives a shell) against the host engine,
with the pairs in any order and only some of them listed, and the metric of such
shells. Tolerance 1e-12 relative to the largest, both sides being sums of the
same terms in FP64."""
import os

import numpy as np
import pytest

from molgw_amd.frontend import Molecule
from molgw_amd.frontend import native as N
from molgw_amd.frontend.basis import BasisSet
from molgw_amd.gw import Engine
from molgw_amd.workloads import upper_pairs

pytestmark = pytest.mark.gpu

BASIS = os.path.join(os.path.dirname(__file__), 'golden', 'basis')
WATER = ['O 0.0 0.0 0.0', 'H 0.757 0.587 0.0', 'H -0.757 0.587 0.0']
CO = ['8 .000000 .000000 .493003', '6 .000000 .000000 -.657337']


@pytest.mark.parametrize('lines, bas, ket, gt', [
    (WATER, 'cc-pVDZ', 'cc-pVDZ', 'PURE'), (CO, 'cc-pVDZ_gaussian', 'cc-pVDZ_gaussian', 'CART'),
    (['C 0 0 0'], 'cc-pVTZ', 'cc-pVTZ', 'PURE'), (['C 0 0 0', 'H 0.6 0.6 0.6'], 'cc-pVDZ', 'cc-pVTZ-RI', 'CART')])
def test_contracted_kets(lines, bas, ket, gt):
    m = Molecule.from_lines(lines)
    bs, ax = BasisSet(m.atoms, m.coords, bas, BASIS, gt), BasisSet(m.atoms, m.coords, ket, BASIS, gt)
    ib = upper_pairs(bs.nbf)
    rng = np.random.default_rng(1)
    ib = ib[:, rng.permutation(ib.shape[1])[:max(1, ib.shape[1] * 2 // 3)]]
    k, l = ib[0] - 1, ib[1] - 1
    ref = N.eri_3center(bs, ax)[k, l, :].copy()
    ref[k == l] *= 0.5
    with Engine(0) as e:
        got = e.eri_3center_ao(bs, ax, ib)
        met = e.eri_2center_ao(ax)
    assert np.max(np.abs(got - ref)) < 1e-12 * np.max(np.abs(ref))
    want = N.eri_2center(ax)
    assert np.max(np.abs(met - want)) < 1e-12 * np.max(np.abs(want))
    np.testing.assert_array_equal(met, met.T)


@pytest.mark.parametrize('natom', [1, 2, 16, 17, 32, 33])
def test_ket_shell_counts(natom):
    # one d shell an atom in the auxiliary basis: at and beside the 16 and 32
    # lanes of ket shells of the (s s| and (p s| kernels
    m = Molecule.from_lines([f'H {0.9 * k} {0.3 * (k % 3)} {0.2 * (k % 2)}' for k in range(natom)])
    bs, ax = (BasisSet(m.atoms, m.coords, b, BASIS, 'PURE') for b in ('cc-pVDZ', 'cc-pVDZ-RI'))
    ib = upper_pairs(bs.nbf)
    k, l = ib[0] - 1, ib[1] - 1
    ref = N.eri_3center(bs, ax)[k, l, :].copy()
    ref[k == l] *= 0.5
    want = N.eri_2center(ax)
    with Engine(0) as e:
        got = e.eri_3center_ao(bs, ax, ib)
        met = e.eri_2center_ao(ax)
    assert np.max(np.abs(got - ref)) < 1e-12 * np.max(np.abs(ref))
    assert np.max(np.abs(met - want)) < 1e-12 * np.max(np.abs(want))
