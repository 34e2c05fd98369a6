"""Engine.trim hands the memory that no context holds back to the device: the
pool's reserved size falls by what the trimmed engine had cached."""
import pytest

from molgw_amd.gw import Engine
from molgw_amd.workloads import synthetic_system

pytestmark = pytest.mark.gpu


def test_trim_gives_the_pool_back():
    s = synthetic_system(130, 420, 20, seed=18, scale=0.3)
    with Engine(0) as eng:
        eng.set_eri_3center(s.eri_3center, s.index_basis, s.nbf)
        eng.set_mo(s.c_matrix, s.energy, s.occupation)
        eng.g0w0(technique='imaginary_pade', nomega_chi_imag=16, nomega_sigma_calc=8)
        held, _ = eng.memory()
        reserved, _ = eng.pool_memory()
        eng.trim()
        kept, _ = eng.memory()
        after, _ = eng.pool_memory()
    assert kept < held <= reserved
    assert after <= reserved - (held - kept) // 2      # the pool rounds its blocks
