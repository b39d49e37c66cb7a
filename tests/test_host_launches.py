"""Which kernels the entry points launch, on the HIP stand-in (no GPU)."""
import pytest

import host_hip
from random_amd import surveys


@pytest.fixture(scope="module")
def stand_in(tmp_path_factory):
    return host_hip.build(tmp_path_factory.mktemp("hip"))


def _line(ns, ncols, nh=1, jobs_x=1):
    return surveys.line2d(nshots=2, nrecv_side=4, ns=ns, ncols=ncols, nscat=1, nh=nh, jobs_x=jobs_x,
                          dh=2000.0 if nh == 1 else 50.0)


def _area(ns, ncols):
    return surveys.area3d(ntr=4, ns=ns, ncols=ncols, nscat=1)


def child_demigrate(hip, cases):
    out = []
    for geometry, ns, ncols, ntr in cases:
        sv = _line(ns, ncols) if geometry == "line" else _area(ns, ncols)
        plan = hip.plan(sv.cfg, sv.ns, sv.dt, sv.vel)
        st, launches, _ = hip.demigrate(plan, ntr)
        names = [k for k, *_ in launches]
        _, (K, W, fast), grid, block, lds = launches[names.index("k_demigrate")]
        assert st == 0 and fast == 0 and block == [512, 1, 1]
        assert 64 * K * W >= ns and lds <= 160 * 1024
        assert names.count("k_demig_finish") == names.count("k_zero_u64") == int(grid[1] > 1)
        out.append(grid[1])
        hip.lib.ktm_plan_destroy(plan)
    return out


def test_demigration_divides_its_columns_only_where_that_pays(stand_in):
    """Calls that parts made slower, and calls that they made several times
    faster, by the measured times of 1 to 16 parts."""
    whole = [("line", ns, 4, n) for ns in (16, 63, 301, 1001, 2001, 5000) for n in (1, 96, 1000, 6000)]
    whole += [("area", ns, 1, n) for ns in (300, 1001) for n in (96, 1000, 4000)]
    whole += [("line", 1001, 16, 3000), ("line", 1001, 60, 6000), ("line", 1501, 60, 6000),
              ("line", 2600, 32, 3000), ("line", 5000, 16, 6000), ("line", 1501, 800, 48000)]
    assert host_hip.run(__file__, stand_in, "child_demigrate", whole) == [1] * len(whole)
    many = [("line", ns, 800, 96) for ns in (63, 300, 1001, 2600, 5000)] + [("area", 751, 61, 3001)]
    assert min(host_hip.run(__file__, stand_in, "child_demigrate", many)) >= 4
