"""Launch counts of the per-launch profiler: every launch of a driver call is
in the counters when the call returns."""
import pytest

from desalm import cases, overset
from desalm.lib import Group, Solver

pytestmark = pytest.mark.gpu

# per pseudo-iteration of a 3-level cycle with 1, 2 and 3 passes: the residual
# of every pass, and the recalc residual of each level's last pass but the
# coarsest's, which is formed once per call
PASSES = (1, 2, 3)


def counts(s, name):
    st = s.profile_stats()
    return [st.get((name, n), (0, 0.0))[0] for n in (1, 2, 3)]


@pytest.mark.parametrize("calls", [1, 2])
def test_counts_of_a_call(gpu, calls):
    itm = 2
    c = cases.wavy(17, 17, 17, ng=3, itm=itm, des=True, iters=PASSES)
    s = Solver(c.params).load_case(c)
    s.profile(True)
    for k in range(1, calls + 1):
        s.mg_driver()
        assert counts(s, "residual") == [k * itm * p for p in PASSES]
        assert counts(s, "residual_recalc") == [k * itm, k * itm, k]
    assert all(ms > 0.0 for _, ms in s.profile_stats().values())
    s.close()


@pytest.mark.parametrize("batched", [True, False])
def test_counts_of_a_group_call(gpu, batched):
    """One launch for all zones counts with zone 1; zone by zone each zone
    counts its own."""
    itm = 2
    cs, tab = overset.hill_blocks([(17, 17, 17), (21, 17, 17)], [0.5], itm=itm, ng=3, iters=PASSES)
    svs = [Solver(c.params).load_case(c) for c in cs]
    g = Group(svs)
    g.set_batched(batched)
    g.set_overset(tab)
    for s in svs:
        s.profile(True)
    g.mg_driver()
    assert counts(svs[0], "residual_recalc") == [itm, itm, 1]
    assert counts(svs[1], "residual_recalc") == ([0, 0, 0] if batched else [itm, itm, 1])
    g.close()
    for s in svs:
        s.close()
