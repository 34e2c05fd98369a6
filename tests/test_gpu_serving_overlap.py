"""Continuous batching with solves that overlap by construction: every solve
waits, its tensor loaded, until the other slots' solves have come as far. (Small
solves take less than a millisecond, so arrival times alone do not make them
overlap.) Each result is the same alone and in the mix."""
import threading

import numpy as np
import pytest

from molgw_amd.serving import Request, Server
from molgw_amd.workloads import alkane_shape, synthetic_system, water_cluster_shape

pytestmark = pytest.mark.gpu
NSLOTS = 3


@pytest.mark.parametrize('technique, precision', [('imaginary_pade', 'bf16x3'), ('imaginary_pade', 'fp16x3'),
                                                  ('imaginary_pade', 'fp64'), ('one_shot', 'fp64')])
def test_overlapping_solves_equal_lone_ones(technique, precision):
    shapes = [alkane_shape(1), water_cluster_shape(1), alkane_shape(2), water_cluster_shape(2), alkane_shape(3),
              water_cluster_shape(3)]
    reqs = [Request(k, synthetic_system(*shape, seed=400 + k, scale=0.3), technique=technique, precision=precision,
                    nomega_chi_imag=16, nomega_sigma_calc=8) for k, shape in enumerate(shapes)]
    with Server(nslots=NSLOTS, hbm_budget=16 << 30) as srv:
        meet = threading.Barrier(NSLOTS, timeout=60)
        for eng in srv.slots:
            def set_mo(*args, _load=eng.set_mo, **kw):
                _load(*args, **kw)
                meet.wait()
            eng.set_mo = set_mo
        mixed = srv.run(reqs, realtime=False)
    spans = sorted((r.start, r.end) for r in mixed)
    for group in (spans[:NSLOTS], spans[NSLOTS:]):
        assert max(s for s, _ in group) < min(e for _, e in group)
    with Server(nslots=1, hbm_budget=16 << 30) as srv:
        alone = [srv.run([r], realtime=False)[0] for r in reqs]
    for a, b in zip(mixed, alone):
        assert a.rid == b.rid
        assert np.max(np.abs(a.energy_qp - b.energy_qp)) <= 1e-10
        assert abs(a.en_rpa - b.en_rpa) <= 1e-10 * max(1.0, abs(b.en_rpa))
