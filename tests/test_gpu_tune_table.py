"""The tuner's table: entries of candidate lists that changed are not taken for
the present ones, and the column tiles of products of few columns are tuned and
looked up like any other."""
import os
import subprocess
import sys

import pytest

from tests.conftest import ROOT

pytestmark = pytest.mark.gpu


def run(code, table):
    pre = ('import sys; sys.path.insert(0, %r)\n'
           'import numpy as np\n'
           'from molgw_amd.gw import Engine, autotune\n'
           'from molgw_amd.workloads import synthetic_system\n') % ROOT
    proc = subprocess.run([sys.executable, '-c', pre + code], env=dict(os.environ, MGW_TUNE_FILE=str(table)),
                          capture_output=True, text=True, timeout=120)
    assert proc.returncode == 0, proc.stderr[-2000:]
    return [list(map(int, line.split())) for line in table.read_text().splitlines() if line.strip()]


# W.B (107): other kernels stood behind its numbers under list 0; the chi0 SYRK
# (105): its default was a 128-wide kernel where 256-wide tiles run now
@pytest.mark.parametrize('family, nomega', [(107, 8), (105, 520)])
def test_entries_of_former_candidate_lists_are_not_used(tmp_path, family, nomega):
    table = tmp_path / 'tune.txt'
    code = ('s = synthetic_system(60, 170, 8, seed=3, scale=0.3)\n'
            'autotune(True)\n'
            'with Engine(0) as e:\n'
            '    e.set_eri_3center(s.eri_3center, s.index_basis, s.nbf)\n'
            '    e.set_mo(s.c_matrix, s.energy, s.occupation)\n'
            '    e.g0w0(technique="imaginary_pade", nomega_chi_imag=%d, nomega_sigma_calc=4, precision="fp16x3")\n'
            % nomega)
    rows = run(code, table)
    mine = [r for r in rows if r[0] == family]
    assert mine
    former = [r[:3] + [0] + r[4:7] + [1] for r in mine]
    table.write_text(''.join(' '.join(map(str, r)) + '\n' for r in [r for r in rows if r[0] != family] + former))
    again = run(code, table)
    assert sorted(r[:7] for r in again[len(rows):]) == sorted(r[:7] for r in mine)


def test_column_tiles_are_tuned(tmp_path):
    """(P|m n) of a window of 16 states runs on column tiles: with tuning on
    they are timed beside the other tiles and recorded, an entry is followed,
    and every candidate gives the same numbers."""
    table = tmp_path / 'tune.txt'
    code = ('s = synthetic_system(177, 371, 9, seed=22, scale=0.3)\n'
            'with Engine(0) as e:\n'
            '    e.set_eri_3center(s.eri_3center, s.index_basis, s.nbf)\n'
            '    e.set_mo(s.c_matrix, s.energy, s.occupation)\n'
            '    ref = e.calculate_eri_3center_mo(1, 177, 2, 17)\n'
            '    e.destroy_eri_3center_mo()\n'
            '    e.set_mo(s.c_matrix, s.energy, s.occupation)\n'
            '    autotune(%s)\n'
            '    for _ in range(2):\n'
            '        got = e.calculate_eri_3center_mo(1, 177, 2, 17)\n'
            '        e.destroy_eri_3center_mo()\n'
            '        e.set_mo(s.c_matrix, s.energy, s.occupation)\n'
            '        assert np.array_equal(got, ref)\n')
    table.touch()
    rows = run(code % 'True', table)
    # class AO2MO, few columns, floor(log2) of 371 x 177, 16 and 177
    key = [0, 0, 0, 2, 16, 4, 7]
    narrow = [r for r in rows if r[:7] == key]
    assert len(narrow) == 1 and 0 <= narrow[0][7] < 4
    for choice in range(4):
        table.write_text(' '.join(map(str, key + [choice])) + '\n')
        run(code % 'False', table)
