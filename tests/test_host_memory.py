"""What the demigration allocates and what it does when memory is short, on
the HIP stand-in (no GPU).  The sums of column parts are the one workspace
that a call can do without."""
import pytest

import host_hip
from random_amd import surveys
from random_amd._lib import KTM_ERR_NOMEM


@pytest.fixture(scope="module")
def stand_in(tmp_path_factory):
    return host_hip.build(tmp_path_factory.mktemp("hip"))


def _plan(hip):
    sv = surveys.line2d(nshots=2, ns=501, ncols=200, nscat=2)
    return hip.plan(sv.cfg, sv.ns, sv.dt, sv.vel)


def _parts(launches):
    """(parts of the columns, finishing launches) of a demigration."""
    names = [k for k, *_ in launches]
    return [launches[names.index("k_demigrate")][2][1] if "k_demigrate" in names else 0,
            names.count("k_demig_finish")]


def _first_call(hip, n, room=None):
    """A new plan's demigration of n traces with that much memory left, then
    the same again, then again with memory: (statuses, parts, bytes)."""
    plan = _plan(hip)
    if room is not None:
        hip.limit(hip.live() + room)
    st, launches, sizes = hip.demigrate(plan, n)
    again = hip.demigrate(plan, n)[0]
    hip.limit()
    after = hip.demigrate(plan, n)[0]
    hip.lib.ktm_plan_destroy(plan)
    return [[st, again, after], _parts(launches), sum(sizes)]


def child_short(hip, n):
    whole = _first_call(hip, n)
    out = [whole, _first_call(hip, n, whole[2] - 1)]
    need = out[1][2]
    return out + [_first_call(hip, n, need), _first_call(hip, n, need - 1)]


def test_a_call_without_memory_for_the_sums_is_not_divided(stand_in):
    n = 1000
    whole, no_sums, least, short = host_hip.run(__file__, stand_in, "child_short", n)
    assert whole[0] == [0, 0, 0] and whole[1][0] > 1 and whole[1][1] == 1
    for r in (no_sums, least):
        assert r[0] == [0, 0, 0] and r[1] == [1, 0]
    assert whole[2] - least[2] == 8 * n * 501
    assert short[0] == [KTM_ERR_NOMEM, KTM_ERR_NOMEM, 0]


def child_give_back(hip, small, large):
    """A divided call, then a larger one, and a block of 16-bit traces, each
    with room for what it needs only if the sums are given back."""
    whole = _first_call(hip, large)[2]
    need = _first_call(hip, large, whole - 1)[2]
    plan = _plan(hip)
    limit = hip.live() + need
    first = hip.demigrate(plan, small)
    hip.limit(limit)
    second = hip.demigrate(plan, large)
    hip.limit()
    hip.lib.ktm_plan_destroy(plan)

    plan = _plan(hip)
    hip.demigrate(plan, small)
    rows = 8 * small * 501 // (4 * hip.lib.ktm_plan_trace_row(plan))
    hip.limit(hip.live())
    decode = hip.migrate(plan, rows, 0, dtype=1)
    third = hip.demigrate(plan, small)
    hip.limit()
    hip.lib.ktm_plan_destroy(plan)
    return [[r[0] for r in (first, second, decode, third)],
            [_parts(r[1]) for r in (first, second, third)]]


def test_the_sums_are_given_back_for_what_a_call_needs(stand_in):
    statuses, parts = host_hip.run(__file__, stand_in, "child_give_back", 1000, 1000000)
    assert statuses == [0, 0, 0, 0]
    assert parts[0][0] > 1 and parts[1:] == [[1, 0], [1, 0]]


def child_no_growth(hip):
    plan = _plan(hip)
    hip.demigrate(plan, 20000)
    return [hip.demigrate(plan, n)[2] for n in (20000, 1000, 130, 1)]


def test_calls_of_no_more_traces_allocate_nothing(stand_in):
    assert host_hip.run(__file__, stand_in, "child_no_growth") == [[], [], [], []]
