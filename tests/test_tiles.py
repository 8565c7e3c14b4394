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
  for (int tiles = 1; tiles <= 300; ++tiles) {
    const int n = awp_cdiv(tiles, AWP_NXCD) * AWP_NXCD;
    for (int r = 0; r < n; ++r) printf("%d %d %d %d\n", tiles, n, r, awp_xcd_in_chunk(r, n));
  }
}
"""


def test_chunk_order_shares_every_chunk_among_the_xcds(tmp_path):
    """Each tile of an i-chunk is one workgroup's, each XCD (workgroup mod 8)
    takes one run of neighbouring tiles, and no XCD more than another plus one
    short run: all of them work on the same planes."""
    table = run_host(tmp_path, ORDER)
    for tiles in range(1, 301):
        _, n, r, t = table[table[:, 0] == tiles].T
        assert len(r) == n[0] and n[0] - tiles < 8
        assert sorted(t) == list(range(n[0]))
        for x in range(8):
            run = t[r % 8 == x]
            assert len(run) == n[0] // 8 and (np.diff(run) == 1).all()
