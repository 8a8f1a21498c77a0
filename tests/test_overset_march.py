"""An overset group marched call after call, as a time-accurate run is."""
import numpy as np
import pytest

from desalm import overset
from desalm.lib import Group, Solver
import pyoracle as po


@pytest.mark.gpu
@pytest.mark.parametrize("batched", [True, False])
def test_group_marched_over_ten_calls_matches_oracle(gpu, batched):
    """The overset workload's hill and Reynolds number on small blocks, ten
    consecutive calls of ten pseudo-iterations, every state carried on."""
    cs, tab = overset.hill_blocks([(25, 17, 13), (29, 21, 13), (33, 17, 17)], [0.35, 0.7], itm=10, amp=0.2,
                                  ren=10595.0, ng=2)
    svs = [Solver(c.params).load_case(c) for c in cs]
    ors = [po.Oracle(c.params).load_case(c) for c in cs]
    g = Group(svs)
    g.set_batched(batched)
    g.set_overset(tab)
    for _ in range(10):
        ig, hg = g.mg_driver()
        io, ho = po.group_mg_driver(ors, tab)
        assert ig == io
        assert np.abs(hg - ho).max() <= 1e-9
        for s, o in zip(svs, ors):
            qg, qo = s.get_state()[0], o.get_state()[0]
            assert max(po.relerr(qg[:, m], qo[:, m]) for m in range(5)) <= 1e-10
    g.close()
    for s in svs:
        s.close()
