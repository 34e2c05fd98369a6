"""The FP16x3 / BF16x3 chi0 build on 256-wide tiles over several K chunks: the
chunks' first slabs and partial tiles, odd and even slab counts, a last chunk of
one, two and three slabs, with and without a last row of half tiles. Each
result equals the 128-wide kernel's bit for bit."""
import numpy as np
import pytest

from molgw_amd.gw import Engine, selfenergy_set_state_range
from molgw_amd.workloads import synthetic_system

pytestmark = pytest.mark.gpu


@pytest.fixture(scope='module')
def eng():
    with Engine(0) as e:
        yield e


def chunks(naux, npole, nomega, cap):
    """Slabs of each K chunk and the 256-wide workgroups of the launch, by the
    rules of split_layout and split_and_syrk (chi0_split.hip)."""
    tm = -(-naux // 128)
    nkt = (-(-npole // 32) + 1) // 2 * 2
    want = max(1, -(-4096 // (tm * (tm + 1) // 2 * nomega)))
    kc = min(max(64, -(-nkt // want)), cap)
    n = [min(kc, nkt - k) for k in range(0, nkt, kc)]
    t256 = tm // 2
    return n, t256 * (t256 + 1) // 2 * len(n) * nomega


# nocc 32: npole = 32 (nbf - 32), so nbf - 32 slabs of 32 transitions
@pytest.mark.parametrize('nbf, cap, slabs, precision', [
    (98, 65, [65, 1], 'fp16x3'), (98, 65, [65, 1], 'bf16x3'), (98, 64, [64, 2], 'fp16x3'), (100, 65, [65, 3], 'fp16x3'),
    (162, 65, [65, 65], 'fp16x3'), (164, 65, [65, 65, 2], 'fp16x3'), (162, 129, [129, 1], 'fp16x3')])
@pytest.mark.parametrize('naux, nomega', [(251, 1370), (379, 690)])
def test_chunked_wide_tiles_equal_narrow_tiles(eng, monkeypatch, nbf, cap, slabs, precision, naux, nomega):
    got_slabs, wide = chunks(naux, 32 * (nbf - 32), nomega, cap)
    assert got_slabs == slabs and wide >= 512
    s = synthetic_system(nbf, naux, 32, seed=21, scale=0.3)
    eng.set_eri_3center(s.eri_3center, s.index_basis, s.nbf)
    eng.set_mo(s.c_matrix, s.energy, s.occupation)
    rng = selfenergy_set_state_range(s.occupation)
    om, wt = np.linspace(0.1, 3.0, nomega), np.ones(nomega)
    monkeypatch.setenv('MGW_CHI_KC_CAP', str(cap))
    got = eng.polarizability_grid(rng, om, wt, precision=precision, return_chi=True)
    monkeypatch.setenv('MGW_CHI_SYRK', '0')
    ref = eng.polarizability_grid(rng, om, wt, precision=precision, return_chi=True)
    assert got[:2] == ref[:2]
    np.testing.assert_array_equal(got[2], ref[2])
    eng.trim()
