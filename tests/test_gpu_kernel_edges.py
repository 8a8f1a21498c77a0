"""Kernels at the sizes where their tiling can go wrong (tile edges,
remainders, the smallest and largest of their range), against the CPU oracle."""
import numpy as np
import pytest

import mlp_oracle as mo
import pyoracle as po
from desalm import cases
from desalm.lib import Solver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nh,m", [(1, 1), (2, 63), (16, 64), (31, 65), (32, 511), (33, 512), (48, 513), (64, 1025)])
def test_mlp_tiles(gpu, nh, m):
    """Forward pass, loss and gradient at the edges of the 64-row tiles, the
    512-row weight-gradient parts and the hidden widths (32: two columns per
    thread, 33: four)."""
    c = cases.wavy(13, 11, 9, ng=2, itm=2, iters=(1, 2))
    s = Solver(c.params).load_case(c)
    s.ws_configure(hidden=nh, samples_per_record=64, capacity=256, seed=3)
    rng = np.random.default_rng(100 * nh + m)
    w = rng.normal(0.0, 0.2, mo.param_count(nh)).astype(np.float32)
    s.ws_params(w)
    x = rng.normal(size=(m, mo.N_IN)).astype(np.float32)
    t = rng.normal(size=(m, 3 * mo.N_COMP)).astype(np.float32)
    w8, x8, t8 = w.astype(np.float64), x.astype(np.float64), t.astype(np.float64)
    y, yo = s.mlp_forward(x), mo.forward(w8, x8, nh)
    # FP32 sums of at most 97 products: 97 roundings of 6e-8 of the largest sum
    assert np.abs(y - yo).max() <= 2e-5 * max(1.0, np.abs(yo).max())
    loss, g = s.mlp_loss_grad(x, t)
    lo, go = mo.loss_grad(w8, x8, t8, nh)
    assert abs(loss - lo) <= 1e-5 * abs(lo)
    # sums over up to 1025 rows, in order: 1025 roundings of 6e-8
    assert np.abs(g - go).max() <= 1e-4 * np.abs(go).max()
    s.close()


@pytest.mark.parametrize("nh,dims", [(1, (5, 5, 5)), (32, (34, 6, 6)), (32, (35, 6, 6)), (33, (18, 6, 6)),
                                     (64, (19, 7, 9))])
def test_learned_start_tiles(gpu, nh, dims):
    """The one-launch learned start with interiors of 27, 512 and 528 nodes on
    128-node tiles (up to 32 hidden units) and 256 and 595 on 64-node tiles."""
    c = cases.wavy(*dims, ng=1, itm=1, seed=9)
    s = Solver(c.params).load_case(c)
    s.ws_configure(hidden=nh, samples_per_record=64, capacity=256, seed=3)
    q, qn, qnm1, _ = s.get_state()
    rng = np.random.default_rng(nh)
    w = rng.normal(0.0, 0.3, mo.param_count(nh)).astype(np.float32)
    stats = np.concatenate([rng.normal(0.0, 0.3, 95), rng.uniform(0.5, 2.0, 95),
                            rng.uniform(0.01, 0.1, 5), np.zeros(5)]).astype(np.float32)
    s.ws_params(w)
    s.ws_stats(stats)
    s.ws_mode(Solver.WS_LEARNED)
    s.set_convergence(0, 0, -8.0, -30.0)
    s.mg_driver()
    got = s.get_state()[0]
    want = mo.warm_start(q, q, qn, qnm1, dims, w.astype(np.float64), nh, stats.astype(np.float64))
    ext = mo.warm_start(q, q, qn, qnm1, dims)
    g = mo.interior_index(dims)
    # the coefficients are FP32 sums of at most 97 products, applied in FP64
    scale = np.abs(want[g] - ext[g]).max(axis=0)
    assert (scale > 0).all()
    assert (np.abs(got[g] - want[g]).max(axis=0) <= 2e-5 * scale + 1e-14).all()
    rest = np.setdiff1d(np.arange(len(q)), g)
    assert np.array_equal(got[rest], q[rest])
    s.close()


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("dims", [(5, 6, 7), (12, 67, 9), (9, 10, 68), (67, 11, 75), (18, 66, 67)])
def test_line_sweep_segments(gpu, dims, prec):
    """Lines of 3 to 73 rows: partial last segments, lines at the change from
    four to eight rows per segment (64 rows), fewer lines than a workgroup
    takes."""
    c = cases.wavy(*dims, ng=1, itm=2, des=True, precision=prec)
    s = Solver(c.params).load_case(c)
    s.mg_driver()
    q, _, _, x = s.get_state()
    o = po.Oracle(c.params).load_case(c)
    o.mg_driver()
    qo, _, _, xo = o.get_state()
    # FP64 sums of a few hundred terms; FP32 solves of dq as a defect correction
    tol = 1e-6 if prec else 1e-10
    assert max(po.relerr(q[:, m], qo[:, m]) for m in range(5)) <= tol
    assert po.relerr(x, xo) <= tol
    assert s.pivot_events == 0
    s.close()


@pytest.mark.parametrize("itk", [1, 3])
@pytest.mark.parametrize("bt", [(1, 8, 6, 1, 3, 2), (4, 8, 1, 6, 6, 2), (3, 2, 4, 0, 4, 4), (0, 1, 6, 6, 1, 6),
                                (5, 3, 5, 4, 5, 0), (2, 0, 0, 3, 6, 6), (7, 7, 1, 4, 7, 7)])
def test_boundary_faces_in_one_launch(gpu, bt, itk):
    """Edge and corner nodes take the i, then j, then k rules in one launch:
    mixed types on adjacent faces, plane copies on one face only (their own
    launches), pinned node on a corner, nu~ below its floor at the start, one
    and three SA sub-iterations (the floor is stored by the last)."""
    c = cases.wavy(11, 9, 13, ng=2, itm=2, des=True, itk=itk, btype=bt, amp=0.02, iters=(1, 2))
    c.params.ifix, c.params.jfix, c.params.kfix = 1, 9, 1
    c.q[::7, 4] = 1e-9
    s = Solver(c.params).load_case(c)
    s.mg_driver()
    q, _, _, x = s.get_state()
    o = po.Oracle(c.params).load_case(c)
    o.mg_driver()
    qo, _, _, xo = o.get_state()
    assert max(po.relerr(q[:, m], qo[:, m]) for m in range(5)) <= 1e-10
    assert po.relerr(x, xo) <= 1e-10
    # the coarsest level's residual, formed once after the last pseudo-iteration
    rh = s.level_field("rh", 2)
    off = o.level_offset(2)
    assert po.relerr(rh, o.get("rh")[off:off + len(rh)]) <= 1e-10
    s.close()


@pytest.mark.parametrize("dims", [(47, 47, 47), (48, 47, 47), (53, 53, 56), (53, 53, 57), (101, 67, 67)])
def test_state_comes_back_through_the_ring(gpu, dims):
    """Read-backs below and above the 4 MiB of a plain copy, one chunk above
    a whole number of 2 MiB chunks and longer than the pinned ring: the state
    that went in comes back, from two threads at once too."""
    import threading
    n = dims[0] * dims[1] * dims[2]
    rng = np.random.default_rng(n)
    c = cases.wavy(*dims, ng=1, itm=1)
    sv = [Solver(c.params) for _ in range(2)]
    st = [[rng.standard_normal((n, 5)) for _ in range(3)] + [rng.standard_normal(n)] for _ in sv]
    for s, a in zip(sv, st):
        s.set_state(*a)
    got = [None, None]

    def read(k):
        got[k] = sv[k].get_state()

    t = [threading.Thread(target=read, args=(k,)) for k in range(2)]
    [x.start() for x in t]
    [x.join() for x in t]
    for a, g in zip(st, got):
        assert all(np.array_equal(u, v) for u, v in zip(a, g))
    for s, a in zip(sv, st):
        assert np.array_equal(s.level_field("q"), a[0])
        s.close()


@pytest.mark.parametrize("noalloc", [False, True])
@pytest.mark.parametrize("n,nsys", [(1, 1), (2, 3), (3, 64), (15, 63), (16, 65), (17, 1), (32, 64), (33, 130),
                                    (97, 7)])
def test_gtsv_chunks(gpu, n, nsys, noalloc):
    """Batched SGTSV at the edges of its 16-row chunks and 64-system waves,
    with interchanges, and zero pivots at the first, an inner and the last
    row."""
    from desalm.lib import gtsv_batch
    rng = np.random.default_rng(1000 * n + nsys)
    dl, d, du, b = (rng.uniform(-1, 1, (nsys, n)) for _ in range(4))
    if nsys >= 3:
        d[1] = dl[1] = 0.0            # INFO 1
        d[2, n // 2] = 0.0
        if n > 1:
            dl[2, n // 2 - 1] = 0.0   # the row before leaves it zero
            dl[2, n // 2] = 0.0
    x, info = gtsv_batch(dl, d, du, b, noalloc=noalloc)
    for s in range(nsys):
        xo, io = po.gtsv(dl[s], d[s], du[s], b[s])
        assert info[s] == io
        if io == 0:
            # a solve of random bands: backward stable, so off by a small
            # multiple of the condition number's share of the largest entry
            assert np.abs(x[s] - xo).max() <= 1e-9 * max(1.0, np.abs(xo).max())
