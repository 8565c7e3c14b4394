import os
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
if str(ROOT) not in sys.path:
    sys.path.insert(0, str(ROOT))


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs the HIP library)")
    config.addinivalue_line("markers", "slow: long CPU test")


@pytest.fixture(scope="session")
def oracle_lib():
    from oracle import oracle
    oracle.load()
    oracle.set_threads(min(4, os.cpu_count() or 1))
    return oracle


# awp_set_tuning's defaults: the launch shapes that a user gets
TUNING = dict(vel_bj=0, str_bj=0, vel_ichunk=0, str_ichunk=0, xcd_remap=1, kw=0, topo_vel_ichunk=0,
              topo_str_ichunk=16, topo_q_ichunk=0, topo_rate_chunk=0, topo_nseg=8, topo_rj=0,
              topo_wsync=1, adj_jgroup=8)


@pytest.fixture
def tuning():
    """Sets launch-shape knobs for one test: they are process-global, and the
    tests after it run the defaults again whether it passed or not."""
    from awp_amd import _lib
    changed = set()

    def put(**knobs):
        for key, value in knobs.items():
            changed.add(key)
            _lib.set_tuning(key, value)

    yield put
    for key in changed:
        _lib.set_tuning(key, TUNING[key])
