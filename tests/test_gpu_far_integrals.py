"""Rounding of the Coulomb integrals at long range, where they have a closed form:
for an s function and a Cartesian function x, xy or xyz (no trace part) that do
not overlap, (s|f) R^(2l+1) / x^l is one constant, and its scatter over distances is
the rounding of the Boys functions F_l and of the prefactors. With every step of
the upward recursion rounded once (a division), the scatter is 0.8, 1.3, 1.8 and
2.5e-16 for l = 0 .. 3; a rounded reciprocal in the place of the division, the
same in every step, gives 0.8, 1.5, 2.1 and 3.1e-16. The bounds lie between."""
import numpy as np
import pytest

from molgw_amd.frontend.basis import BasisSet
from molgw_amd.gw import Engine

pytestmark = pytest.mark.gpu


def components(l):
    return [(l - i, i - k, k) for i in range(l + 1) for k in range(i + 1)]


@pytest.mark.parametrize('powers, bound', [((0, 0, 0), 1.0e-16), ((1, 0, 0), 1.4e-16), ((1, 1, 0), 1.93e-16),
                                           ((1, 1, 1), 2.75e-16)])
def test_scatter_of_the_multipole_law(tmp_path, powers, bound):
    (tmp_path / 'H_far').write_text('4\n' + ''.join(f'1 {l}\n 1.0 1.0\n' for l in range(4)))
    n, l = 60, sum(powers)
    first = np.cumsum([0] + [len(components(k)) for k in range(4)])
    column = first[l] + components(l).index(powers)
    z = np.cumsum(8.0 + 2.0 * np.random.default_rng(l).random(n))
    xyz = np.outer(z, powers if l else (1, 0, 0)).astype(float)
    with Engine(0) as eng:
        m = eng.eri_2center_ao(BasisSet([1] * n, xyz, 'far', str(tmp_path), 'CART'))
    x = np.abs(z[None, :].astype(np.longdouble) - z[:, None])
    r2 = x * x * max(1, l)
    # T = R^2 / 2 from 40, where the functions' overlap has gone, to 2e4
    far = (r2 > 80.0) & (r2 < 4.0e4)
    v = np.abs(m[0::first[-1], column::first[-1]][far]).astype(np.longdouble) * r2[far] ** (l + np.longdouble(0.5)) / x[far] ** l
    scatter = float(np.sqrt(np.mean((v / v.mean() - 1.0) ** 2)))
    assert len(v) > 1000 and scatter <= bound
