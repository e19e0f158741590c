"""The index check of the 3D tiles with the columns beside a tile (lanes -1 and 64) and the rows around it that the fused
kernel reads, at extents next to multiples of its 64 z cells and 14 rows."""
import os
import shutil
import subprocess

from tests.test_tile_index_3d import CHECKER, CSRC

SHAPES = [  # (nx, ny, nz, periodic x, y, z, planes per tile)
    (5, 13, 63, 0, 0, 0, 2), (5, 14, 64, 0, 0, 0, 5), (5, 15, 65, 0, 0, 0, 16), (4, 27, 127, 1, 1, 1, 3),
    (4, 28, 128, 1, 1, 1, 4), (4, 29, 129, 1, 1, 1, 32), (33, 2, 2, 0, 1, 1, 16), (2, 14, 3, 0, 0, 1, 1),
    (3, 1, 192, 0, 1, 0, 2), (16, 43, 5, 0, 1, 1, 16),
]


def test_columns_beside_a_tile_stay_in_the_grid(tmp_path):
    checker = CHECKER.replace('for (int lane = 0; lane < kLanes; ++lane)', 'for (int lane = -1; lane <= kLanes; ++lane)')
    checker = checker.replace('r < kRows + 2;', 'r < kRows + 3;')
    assert checker.count('lane = -1') == 1 and checker.count('kRows + 3') == 1
    (tmp_path / 'check.cpp').write_text(checker)
    binary = tmp_path / 'check'
    compiler = shutil.which('g++') or shutil.which('c++')
    subprocess.run([compiler, '-std=c++17', '-O1', f'-I{CSRC}', os.path.join(tmp_path, 'check.cpp'), '-o', str(binary)],
                   check=True)
    result = subprocess.run([str(binary), *(str(v) for s in SHAPES for v in s)], capture_output=True, text=True)
    assert result.returncode == 0, result.stdout
    assert f'checked {len(SHAPES)} cases, 0 failures' in result.stdout
