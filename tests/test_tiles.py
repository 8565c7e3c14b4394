"""The tile and march rules of the Cartesian kernels, compiled for the host:
every level and row of a column is some lane's, exactly one's, and the lanes
that a tile leaves idle are those its rule allows."""
import os
import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest

ROOT = Path(__file__).resolve().parents[1]
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
NMAX = 700
PROGRAM = r"""
#include <stdio.h>
#include <stdlib.h>
#include "awp_common.h"
#include "awp_tuning.h"
int main() {
  for (int n = 1; n <= %d; ++n)
    for (int rule = 0; rule < 3; ++rule) {
      const AwpTile t = rule == 2 ? awp_pick_full_tile(n, 0) : awp_pick_tile(n, rule == 1, 0, 0);
      int wrong = 0;
      for (int l = 0; l < 64 * t.waves; ++l) wrong += (l * t.mul >> 20) != l / t.width;
      printf("%%d %%d %%d %%d %%d %%d %%d\n", rule, n, t.width, t.rows, t.waves, t.nkt, wrong);
    }
}
""" % NMAX


def run_host(tmp_path, program):
    """Compile a host program against the library's headers; its output."""
    if not Path(HIPCC).exists() and shutil.which("hipcc") is None:
        pytest.skip("no hipcc")
    src, exe = tmp_path / "rules.hip", tmp_path / "rules"
    src.write_text(program)
    subprocess.run([HIPCC, "--offload-host-only", "-std=c++17", "-O1", "-I",
                    str(ROOT / "awp_amd" / "csrc"), str(src), "-o", str(exe)], check=True,
                   capture_output=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout
    return np.array([[int(x) for x in line.split()] for line in out.splitlines()])


@pytest.fixture(scope="module")
def tiles(tmp_path_factory):
    return run_host(tmp_path_factory.mktemp("tiles"), PROGRAM)


def test_tiles_cover_the_column(tiles):
    rule, n, width, rows, waves, nkt, wrong = tiles.T
    assert (wrong == 0).all()
    assert (rows >= 1).all() and (waves >= 1).all() and (waves <= 8).all()
    assert (rows * width <= 64 * waves).all()
    assert (nkt * width >= n).all() and ((nkt - 1) * width < n).all()


def test_short_columns_keep_their_lanes(tiles):
    """Columns of up to 32 levels, and of 65 to 96 in 16-bit storage, leave no
    more lanes idle than runs of 32 levels."""
    for rule, n, width, rows, waves, nkt, _ in tiles:
        if (rule < 2 and n <= 32) or (rule == 1 and 64 < n <= 96):
            assert 64 * waves * nkt <= 32 * -(-n // 32) * rows, (n, width, rows, waves)


def test_plasticity_workgroups_fill_the_simds(tiles):
    """drprecpc_calc runs four waves per SIMD: no workgroup of 5, 6 or 7 waves,
    and no more lanes idle than in runs of 64 levels."""
    for rule, n, width, rows, waves, nkt, _ in tiles:
        if rule == 2:
            assert waves in (1, 2, 3, 4, 8), (n, waves)
            assert 64 * waves * nkt <= 64 * -(-n // 64) * rows, (n, width, rows, waves)


ORDER = r"""
#include <stdio.h>
#include "awp_common.h"
int main() {
  for (int n = 1; n <= 300; ++n)
    for (int b = 0; b < n; ++b) printf("%d %d %d\n", n, b, awp_xcd_remap(b, n));
}
"""


def test_xcds_share_the_blocks_in_runs(tmp_path):
    """n blocks (a launch's or one i-chunk's): each tile is one block's, each
    XCD (block mod 8) takes one run of neighbouring tiles, and the runs differ
    by one tile at most."""
    table = run_host(tmp_path, ORDER)
    for n in range(1, 301):
        _, b, t = table[table[:, 0] == n].T
        assert sorted(t) == list(range(n))
        runs = [t[b % 8 == x] for x in range(8)]
        assert all((np.diff(r) == 1).all() for r in runs)
        assert max(map(len, runs)) - min(map(len, runs)) <= 1
