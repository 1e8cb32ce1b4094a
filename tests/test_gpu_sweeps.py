"""GPU parity of the sweeps that pick nodes by hat masks, at the edges of their
windows (64 nodes), groups of eight and sixteen nodes, blocks (64 points) and
dof tiles (32), and on both sides of every rule that chooses between them.

Every subset of a grid's nodes is a state, so rows drawn at random give any
number of nodes and paths whose prefixes are no nodes. Tolerance: each of the
nno terms B_k S_k is rounded a few times, to 53 bits (FP64) or 22 (the split
of F16X2, the coarsest), of a term no larger than B_k max|S|: 1e-12 and 1e-6 of
max_p sum_k B_k max|S| leave more than an order of magnitude for up to 2,000
terms in FP64, and for the sums over them in FP32.
"""
import numpy as np
import pytest

import hddm_lb
import oracle
from gpu_util import ALL_PRECISIONS, TOL, run_forward

pytestmark = pytest.mark.gpu

# dim, base, depth, probability, nodes of the grid; nodes drawn (0: all); dofs; points
CASES = [
    (6, 3, 5, 0.0, 0, 1, 1, 1),
    (6, 3, 5, 0.0, 0, 63, 31, 63),
    (6, 3, 5, 0.0, 0, 64, 32, 64),
    (6, 3, 5, 0.0, 0, 65, 33, 65),
    (16, 2, 6, 0.3, 6000, 127, 96, 129),
    (16, 2, 6, 0.3, 6000, 1009, 128, 700),
    (16, 2, 6, 0.3, 6000, 1600, 160, 130),
    (32, 2, 5, 0.3, 4000, 1024, 40, 200),
    (59, 3, 4, 0.0, 0, 1500, 65, 100),      # more hats than the table in LDS takes
    (10, 0, 0, 0.0, 0, 1700, 20, 90),       # up to ten factors a node
]


@pytest.mark.parametrize("halves", [False, True])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "d%d-n%d-c%d-p%d" % (c[0], c[5], c[6], c[7]))
def test_node_subsets(case, halves):
    dim, base, depth, p, nodes, pick, dofs, npts = case
    r = np.random.default_rng(pick)
    if depth:
        ii, jj, lv, ix = hddm_lb.generate_grid(dim, base, depth, p, 7, nodes)
    else:
        hats = np.array([(0, 0), (2, 0), (2, 2), (4, 1), (4, 3)], np.int32)
        picks = np.unique(r.integers(0, len(hats), (4 * pick, dim)) * (r.random((4 * pick, dim)) < 0.5), axis=0)
        ii, jj = hats[picks, 0], hats[picks, 1]
    rows = np.sort(r.choice(ii.shape[0], min(pick, ii.shape[0]), replace=False))
    ii, jj = np.ascontiguousarray(ii[rows]), np.ascontiguousarray(jj[rows])
    if halves:
        # an index_i that is no power of two: these states keep the walking sweeps
        ii, jj = np.where(ii > 1, 3 * ii, ii).astype(ii.dtype), np.where(ii > 1, 3 * jj, jj).astype(jj.dtype)
    S = r.standard_normal((len(rows), dofs))
    X = hddm_lb.synthetic_points(npts, dim, 9)
    X[0] = 0.5
    if npts > 2:
        X[1], X[2] = 0.0, 1.0
    yo = oracle.forward(ii, jj, S, X)
    den = oracle.forward(ii, jj, np.ones((len(rows), 1)), X).max() * np.abs(S).max()
    c = hddm_lb.Context(0)
    c.upload_state(0, ii, jj, S)
    for prec in ALL_PRECISIONS:
        print("nodes", len(rows), "precision", prec, flush=True)
        y = run_forward(c, X, precision=prec)
        err = np.abs(y - yo).max() / max(den, 1e-300)
        print("  error", err, flush=True)
        assert err <= TOL[prec]
    c.close()


# dim, base, depth, probability, nodes of the grid; nodes drawn; dofs; points
ADJOINT_CASES = [
    (6, 3, 5, 0.0, 0, 1, 1, 1),
    (6, 3, 5, 0.0, 0, 15, 16, 63),
    (6, 3, 5, 0.0, 0, 17, 17, 64),
    (6, 3, 5, 0.0, 0, 65, 31, 65),
    (16, 2, 6, 0.3, 6000, 1009, 32, 700),
    (17, 2, 5, 0.3, 4000, 1024, 5, 129),
    (32, 2, 5, 0.3, 4000, 1500, 32, 200),
    (10, 0, 0, 0.0, 0, 700, 20, 90),        # up to ten factors a node: the per-tile kernels
]


@pytest.mark.parametrize("case", ADJOINT_CASES, ids=lambda c: "d%d-n%d-c%d-p%d" % (c[0], c[5], c[6], c[7]))
def test_adjoint_node_subsets(case):
    """The default adjoint against the per-tile kernels' walk, at kinks too:
    both sum the same FP64 terms in another order (1e-12 normwise for dS, whose
    terms are products of a basis value in [0, 1] and g; 1e-10 for dx, whose
    terms carry 1 / phi). dx is bitwise the same on every call."""
    import torch
    dim, base, depth, p, nodes, pick, dofs, npts = case
    r = np.random.default_rng(pick)
    if depth:
        ii, jj, lv, ix = hddm_lb.generate_grid(dim, base, depth, p, 7, nodes)
    else:
        hats = np.array([(0, 0), (2, 0), (2, 2), (4, 1), (4, 3)], np.int32)
        picks = np.unique(r.integers(0, len(hats), (4 * pick, dim)) * (r.random((4 * pick, dim)) < 0.5), axis=0)
        ii, jj = hats[picks, 0], hats[picks, 1]
    rows = np.sort(r.choice(ii.shape[0], min(pick, ii.shape[0]), replace=False))
    ii, jj = np.ascontiguousarray(ii[rows]), np.ascontiguousarray(jj[rows])
    S = r.standard_normal((len(rows), dofs))
    X = hddm_lb.synthetic_points(npts, dim, 9)
    X[0] = 0.5
    if npts > 4:
        X[1], X[2], X[3], X[4] = 0.0, 1.0, 1e-20, 0.25
    x = torch.from_numpy(X).cuda()
    g = torch.from_numpy(r.standard_normal((npts, dofs))).cuda()
    c = hddm_lb.Context(0)
    c.upload_state(0, ii, jj, S)
    got = []
    for form in (1, 0, 0):
        c.set_option(hddm_lb.OPT_FORMULATION, form)
        dx = torch.full((npts, dim), np.nan, dtype=torch.float64, device="cuda")
        ds = torch.full((len(rows) * dofs,), np.nan, dtype=torch.float64, device="cuda")
        print("nodes", len(rows), "formulation", form, flush=True)
        c.adjoint(x, g, dx, ds, None, hddm_lb.FP64)
        torch.cuda.synchronize()
        assert c.device_status() == 0
        got.append((dx.cpu().numpy(), ds.cpu().numpy()))
    c.close()
    (dx1, ds1), (dx0, ds0), (dxr, _) = got
    err = [np.abs(a - b).max() / max(np.abs(b).max(), 1e-300) for a, b in ((dx0, dx1), (ds0, ds1))]
    print("  errors", err, flush=True)
    assert err[0] <= 1e-10 and err[1] <= 1e-12
    assert np.array_equal(dx0, dxr)


@pytest.mark.parametrize("npts", [1, 63, 1023, 1025, 2047, 2048, 2049])
@pytest.mark.parametrize("sort", [0, 1])
def test_point_order_and_plan_of_small_batches(npts, sort):
    """Both sides of the size up to which one workgroup orders the points and
    plans the items: three states, rows of an unknown state untouched."""
    dim, dofs = 6, 8
    r = np.random.default_rng(npts)
    c = hddm_lb.Context(0)
    c.set_option(hddm_lb.OPT_SORT_POINTS, sort)
    states = []
    for s in range(3):
        ii, jj, lv, ix = hddm_lb.generate_grid(dim, 2, 4, 0.5, 11 + s, 300)
        S = r.standard_normal((ii.shape[0], dofs))
        c.upload_state(s, ii, jj, S)
        states.append((ii, jj, S))
    X = hddm_lb.synthetic_points(npts, dim, 5)
    sid = r.integers(0, 4, npts).astype(np.int32)
    print("points", npts, "sort", sort, flush=True)
    y = run_forward(c, X, sid, hddm_lb.FP64)
    c.close()
    assert np.isnan(y[sid == 3]).all()
    for s, (ii, jj, S) in enumerate(states):
        at = sid == s
        if at.any():
            den = oracle.forward(ii, jj, np.ones((len(S), 1)), X[at]).max() * np.abs(S).max()
            assert np.abs(y[at] - oracle.forward(ii, jj, S, X[at])).max() <= 1e-12 * den
