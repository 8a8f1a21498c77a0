"""Infinite physical time step: every 1.5 dtau / delti and x / (2 delti J)
term is zero, so a step is the steady one of the same fields.  The FP64 line
sweeps' own division has to return that zero as IEEE division does."""
import math

import numpy as np
import pytest

from desalm import cases
from desalm.lib import Solver
import pyoracle as po


def case(des, unsteady, **kw):
    c = cases.wavy(19, 17, 13, ng=1, itm=2, des=des, seed=5, **kw)
    c.params.delti = math.inf
    c.params.unsteady = int(unsteady)
    return c


@pytest.mark.parametrize("des", [False, True])
@pytest.mark.parametrize("unsteady", [False, True])
def test_oracle_takes_an_infinite_time_step(des, unsteady):
    o = po.Oracle(case(des, unsteady).params).load_case(case(des, unsteady))
    o.mg_driver()
    assert all(np.all(np.isfinite(a)) for a in o.get_state())


@pytest.mark.gpu
@pytest.mark.parametrize("des", [False, True])
@pytest.mark.parametrize("unsteady", [False, True])
@pytest.mark.parametrize("prec", [0, 1])
def test_infinite_time_step(gpu, des, unsteady, prec):
    c = case(des, unsteady, precision=prec)
    s = Solver(c.params).load_case(c)
    s.mg_driver()
    q, _, _, x = s.get_state()
    o = po.Oracle(c.params).load_case(c)
    o.mg_driver()
    qo, _, _, xo = o.get_state()
    tol = 1e-6 if prec else 1e-10  # FP32 solves of dq as a defect correction
    assert max(po.relerr(q[:, m], qo[:, m]) for m in range(5)) <= tol
    assert po.relerr(x, xo) <= tol
    assert s.pivot_events == 0
    s.close()
