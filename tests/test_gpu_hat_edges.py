"""GPU tests of the kernels over hat masks where values leave the ordinary:
coordinates of -0.0, surpluses and gradients that are not finite.
"""
import numpy as np
import pytest

import hddm_lb
import oracle

pytestmark = pytest.mark.gpu


def adjoint(c, X, G):
    import torch
    x, g = torch.from_numpy(X).cuda(), torch.from_numpy(G).cuda()
    dx = torch.full(X.shape, np.nan, dtype=torch.float64, device="cuda")
    ds = torch.full((c.surplus_offset(-1)[1],), np.nan, dtype=torch.float64, device="cuda")
    c.adjoint(x, g, dx, ds, None, hddm_lb.FP64)
    torch.cuda.synchronize()
    return dx.cpu().numpy(), ds.cpu().numpy()


@pytest.mark.parametrize("dim,dofs", [(6, 5), (20, 32)])
def test_adjoint_at_negative_zero(dim, dofs):
    """A hat (i, 0) has its peak at 0 of either sign: its slope there is 0, as
    the oracle's. dx of the same points at +0.0 and -0.0 is the same, bit for bit."""
    ii, jj, lv, ix = hddm_lb.generate_grid(dim, 3 if dim < 10 else 2, 5, 0.0, 1, 0)
    assert ((ii > 0) & (jj == 0)).any()
    r = np.random.default_rng(dim)
    S = r.standard_normal((len(ii), dofs))
    X = hddm_lb.synthetic_points(130, dim, 4)
    at = r.random(X.shape) < 0.3
    at[0] = True
    G = r.standard_normal((130, dofs))
    c = hddm_lb.Context(0)
    c.upload_state(0, ii, jj, S)
    got = []
    for zero in (0.0, -0.0):
        X[at] = zero
        print("dim", dim, "zero", zero, flush=True)
        got.append(adjoint(c, X, G)[0])
    c.close()
    dxo = oracle.adjoint(ii, jj, S, X, G)[0]
    # as the adjoint's parity tests: dx to 1e-10 normwise
    for dx in got:
        assert np.abs(dx - dxo).max() <= 1e-10 * np.abs(dxo).max()
    assert np.array_equal(got[0], got[1])


# dim, base, depth, nodes of the grid (0: all), dofs: hat tables of one tile and
# of two; more hats than those take, one tile and three
GRIDS = [(6, 3, 4, 0, 20), (16, 2, 6, 6000, 40), (4, 7, 8, 0, 8), (59, 3, 4, 0, 65)]


@pytest.mark.parametrize("npts", [1, 3, 200])
@pytest.mark.parametrize("grid", GRIDS, ids=lambda g: "d%d-c%d" % (g[0], g[4]))
def test_nodes_that_no_point_meets_do_not_count(grid, npts):
    """Surpluses of nodes outside every point's block leave the results alone
    whatever they are: infinite and NaN ones give the results of zeros, bit for
    bit, forward and dx."""
    import torch
    dim, base, depth, nodes, dofs = grid
    ii, jj, lv, ix = hddm_lb.generate_grid(dim, base, depth, 0.3 if nodes else 0.0, 7, nodes)
    r = np.random.default_rng(npts)
    if len(ii) > 8000:
        rows = np.sort(r.choice(len(ii), 6000, replace=False))
        ii, jj = np.ascontiguousarray(ii[rows]), np.ascontiguousarray(jj[rows])
    # supports in the lower half of the first dimension
    low = (ii[:, 0] > 0) & (jj[:, 0] + 1 <= ii[:, 0] // 2)
    assert low.sum() > 5
    S = r.standard_normal((len(ii), dofs))
    X = hddm_lb.synthetic_points(npts, dim, 9)
    X[:, 0] = 0.5 + 0.5 * X[:, 0]
    G = r.standard_normal((npts, dofs))
    x = torch.from_numpy(X).cuda()
    c = hddm_lb.Context(0)
    got = []
    for bad in (0.0, np.inf, np.nan):
        S[low] = bad
        S[np.flatnonzero(low)[::2]] *= -1.0
        c.upload_state(0, ii, jj, S)
        res = []
        for prec in (hddm_lb.FP64, hddm_lb.F32):
            print("dim", dim, "points", npts, "surplus", bad, "precision", prec, flush=True)
            y = torch.full((npts, dofs), np.nan, dtype=torch.float64, device="cuda")
            c.forward(x, y, None, prec)
            torch.cuda.synchronize()
            res.append(y.cpu().numpy())
        if dim <= 32 and dofs <= 32:
            res.append(adjoint(c, X, G)[0])
        got.append(res)
    c.close()
    for a in got:
        for p, q in zip(a, got[0]):
            assert np.isfinite(p).all() and np.array_equal(p, q)


def test_infinite_gradient_at_prefixes_that_are_no_nodes():
    """A prefix that is no node has no surplus and adds nothing, also to the dx
    of a point whose upstream gradient is infinite."""
    r = np.random.default_rng(3)
    dim, dofs = 8, 4
    on = np.unique(r.random((200, dim)) < 0.4, axis=0)
    # products of hats (2, 2), whose slope is +2 at every point below 1; those of
    # even size only, so that every other prefix is none
    on = on[on.sum(1) % 2 == 0]
    on = on[(on.sum(1) >= 2) & (on.sum(1) <= 6)]
    ii = np.where(on, 2, 0).astype(np.int32)
    jj = ii.copy()
    S = 1.0 + r.random((len(ii), dofs))
    X = 0.6 + 0.3 * r.random((5, dim))
    G = 1.0 + r.random((5, dofs))
    G[2, 1] = np.inf
    c = hddm_lb.Context(0)
    c.upload_state(0, ii, jj, S)
    dx, ds = adjoint(c, X, G)
    c.close()
    dxo = oracle.adjoint(ii, jj, S, X, G)[0]
    assert np.array_equal(np.isinf(dxo[2]), on.any(0)) and np.array_equal(dx[2], dxo[2])
    rest = [0, 1, 3, 4]
    assert np.abs(dx[rest] - dxo[rest]).max() <= 1e-10 * np.abs(dxo[rest]).max()


def test_host_calls_do_not_depend_on_what_is_queued_with_them():
    """Small host calls of several threads are run as one batch; each gives the
    bits of the call made alone, however many were queued."""
    import threading
    dim, dofs, n, nthreads = 16, 12, 60, 16
    ii, jj, lv, ix = hddm_lb.generate_grid(dim, 2, 7, 0.3, 7, 60000)
    c = hddm_lb.Context(0)
    c.upload_state(0, ii, jj, np.random.default_rng(1).standard_normal((len(ii), dofs)))
    X = [hddm_lb.synthetic_points(n, dim, 20 + t) for t in range(nthreads)]
    alone = [c.forward_host(x, np.zeros((n, dofs)), None, hddm_lb.FP64).copy() for x in X]
    bad = []

    def worker(t):
        for k in range(20):
            if not np.array_equal(c.forward_host(X[t], np.zeros((n, dofs)), None, hddm_lb.FP64), alone[t]):
                bad.append((t, k))
    before = c.host_call_stats()
    th = [threading.Thread(target=worker, args=(t,)) for t in range(nthreads)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    after = c.host_call_stats()
    print("requests", after[0] - before[0], "batches", after[1] - before[1], "different", len(bad), flush=True)
    c.close()
    assert not bad


# dim, base, depth, probability, nodes of the grid (0: all), dofs: hat tables of
# one tile and of four; direct, one tile and more than four
BATCH_GRIDS = [(16, 2, 6, 0.3, 20000, 24), (24, 1, 6, 0.3, 12000, 128), (6, 6, 7, 0.0, 0, 8), (59, 2, 4, 0.0, 0, 150)]


@pytest.mark.parametrize("grid", BATCH_GRIDS, ids=lambda g: "d%d-c%d" % (g[0], g[5]))
def test_results_in_batches_of_other_sizes(grid):
    """A point's forward has the same bits in every batch of up to 64 points,
    and in one of the same size made as a plan or without allocations. Batches
    of other sizes may share out a state's nodes in other runs: the same terms
    in another order, to the tolerances of any order (1e-12 and 1e-6)."""
    import torch
    dim, base, depth, p, nodes, dofs = grid
    r = np.random.default_rng(dim)
    c = hddm_lb.Context(0)
    for s, keep in enumerate((1.0, 0.4)):
        ii, jj, lv, ix = hddm_lb.generate_grid(dim, base, depth, p, 7, nodes)
        rows = np.flatnonzero(r.random(len(ii)) < keep)
        c.upload_state(s, np.ascontiguousarray(ii[rows]), np.ascontiguousarray(jj[rows]), r.standard_normal((len(rows), dofs)))
    big = 40000
    x = torch.from_numpy(hddm_lb.synthetic_points(big, dim, 9)).cuda()
    sid = torch.from_numpy(r.integers(0, 2, big).astype(np.int32)).cuda()

    def run(n, prec):
        y = torch.full((n, dofs), np.nan, dtype=torch.float64, device="cuda")
        c.forward(x[:n], y, sid[:n], prec)
        torch.cuda.synchronize()
        return y
    for prec in (hddm_lb.FP64, hddm_lb.F32):
        ref, one = run(big, prec), run(64, prec)
        for n in (1, 7, 64, 700, 3000, 13000):
            print("dim", dim, "precision", prec, "points", n, flush=True)
            a = run(n, prec)
            if n <= 64:
                assert torch.equal(a, one[:n])
            assert (a - ref[:n]).abs().max() <= (1e-12 if prec == hddm_lb.FP64 else 1e-6) * ref.abs().max()
            if n in (64, 3000):
                b = torch.full_like(a, np.nan)
                assert hddm_lb.lib.hddm_lb_forward_noalloc(c._h, n, x.data_ptr(), dim, sid.data_ptr(), b.data_ptr(), dofs,
                                                           prec, torch.cuda.current_stream().cuda_stream) == 0
                torch.cuda.synchronize()
                d = torch.full_like(a, np.nan)
                plan = c.plan(x[:n], d, sid[:n], prec)
                plan.launch(torch.cuda.current_stream())
                torch.cuda.synchronize()
                assert torch.equal(b, a) and torch.equal(d, a)
                del plan
    c.close()


def test_last_config_gives_the_waves_of_the_kernel_that_ran():
    import torch
    # (grid, formulation) and the waves in FP64 and F32: hat tables, direct, walking
    for (dim, base, depth, form), waves in (((6, 3, 4, 0), (8, 12)), ((4, 7, 8, 0), (8, 8)), ((6, 3, 4, 1), (4, 4))):
        c = hddm_lb.Context(0)
        ii, jj, lv, ix = hddm_lb.generate_grid(dim, base, depth, 0.0, 7, 0)
        c.upload_state(0, ii, jj, np.ones((len(ii), 8)))
        c.set_option(hddm_lb.OPT_FORMULATION, form)
        x = torch.full((100, dim), 0.3, dtype=torch.float64, device="cuda")
        y = torch.zeros((100, 8), dtype=torch.float64, device="cuda")
        for prec, want in zip((hddm_lb.FP64, hddm_lb.F32), waves):
            print("dim", dim, "formulation", form, "precision", prec, flush=True)
            c.forward(x, y, None, prec)
            torch.cuda.synchronize()
            assert c.last_config()["waves"] == want
        c.close()


@pytest.mark.parametrize("hats,waves", [(510, 8), (511, 8), (2046, 8), (2047, 4), (12000, 4)])
def test_number_of_hats(hats, waves):
    """Up to 2,046 distinct hats a state runs on the sweeps over hat masks, past
    that on the walking ones, also where the table that lists them is full."""
    dim, dofs = 60, 9
    every = [(d, 2 ** k, j) for k in range(1, 10) for d in range(dim) for j in range(0 if k == 1 else 1, 2 ** k + (k == 1), 1 if k == 1 else 2)]
    every = [(d, i, j) for d, i, j in every if not (i == 2 and j == 1)]
    r = np.random.default_rng(hats)
    pick = every[:hats]
    assert len(set(pick)) == hats
    # the root, a node of one factor each, and pairs of them
    ii, jj = np.zeros((1 + hats + 300, dim), np.int32), np.zeros((1 + hats + 300, dim), np.int32)
    for n, (d, i, j) in enumerate(pick):
        ii[1 + n, d], jj[1 + n, d] = i, j
    for n in range(300):
        for d, i, j in (pick[k] for k in r.choice(hats, 2, replace=False)):
            ii[1 + hats + n, d], jj[1 + hats + n, d] = i, j
    S = r.standard_normal((len(ii), dofs))
    X = hddm_lb.synthetic_points(150, dim, 9)
    import torch
    c = hddm_lb.Context(0)
    c.upload_state(0, ii, jj, S)
    x = torch.from_numpy(X).cuda()
    y = torch.full((150, dofs), np.nan, dtype=torch.float64, device="cuda")
    print("hats", hats, flush=True)
    c.forward(x, y, None, hddm_lb.FP64)
    torch.cuda.synchronize()
    got = c.last_config()["waves"]
    c.close()
    yo = oracle.forward(ii, jj, S, X)
    den = oracle.forward(ii, jj, np.ones((len(ii), 1)), X).max() * np.abs(S).max()
    assert got == waves
    assert np.abs(y.cpu().numpy() - yo).max() <= 1e-12 * den


def test_tuned_forward_after_coalesced_calls():
    """The tuner's choice for a size is used by calls of that size however they
    share out nodes: a batch of queued host calls, then device batches."""
    import threading
    import torch
    dim, dofs, n = 16, 12, 64
    ii, jj, lv, ix = hddm_lb.generate_grid(dim, 2, 7, 0.3, 7, 60000)
    S = np.random.default_rng(1).standard_normal((len(ii), dofs))
    c = hddm_lb.Context(0)
    c.set_option(hddm_lb.OPT_AUTOTUNE, 1)
    c.upload_state(0, ii, jj, S)
    X = hddm_lb.synthetic_points(16 * n, dim, 20)
    yo = oracle.forward(ii, jj, S, X)
    out = np.zeros((16 * n, dofs))

    def worker(t):
        for k in range(5):
            out[t * n:(t + 1) * n] = c.forward_host(X[t * n:(t + 1) * n], np.zeros((n, dofs)), None, hddm_lb.FP64)
    th = [threading.Thread(target=worker, args=(t,)) for t in range(16)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    print("coalesced", flush=True)
    assert np.abs(out - yo).max() <= 1e-12 * np.abs(yo).max()
    for m in (1024, 512, 900):
        x = torch.from_numpy(X[:m]).cuda()
        y = torch.zeros((m, dofs), dtype=torch.float64, device="cuda")
        print("points", m, flush=True)
        c.forward(x, y, None, hddm_lb.FP64)
        torch.cuda.synchronize()
        assert np.abs(y.cpu().numpy() - yo[:m]).max() <= 1e-12 * np.abs(yo).max()
    c.close()


# dim, base, depth, nodes of the grid (0: all), dofs, points of the large batch,
# whether that walks; direct sweep and hat tables
DENSE = [(4, 7, 8, 0, 8, 300000, True), (3, 6, 7, 0, 40, 1 << 20, True), (8, 1, 6, 2000, 8, 1 << 20, True),
         (8, 1, 6, 2000, 8, 65536, False), (16, 2, 6, 6000, 40, 100000, False)]


@pytest.mark.parametrize("grid", DENSE, ids=lambda g: "d%d-c%d-p%d" % (g[0], g[4], g[5]))
def test_large_batches_in_few_dimensions(grid):
    """Batches whose blocks meet few of a state's nodes run on the walking sweep;
    its results are those of the other sweeps up to rounding (1e-12, 1e-6), for
    every precision, with padded rows, two states and points of none."""
    import torch
    dim, base, depth, nodes, dofs, n, walks = grid
    r = np.random.default_rng(dim)
    c = hddm_lb.Context(0)
    most = 0.0
    for s, nd in enumerate((dofs, max(1, dofs // 2))):
        ii, jj, lv, ix = hddm_lb.generate_grid(dim, base, depth, 0.3 if nodes else 0.0, 7, nodes)
        S = r.standard_normal((len(ii), nd))
        most = max(most, oracle.forward(ii, jj, np.ones((len(ii), 1)), r.random((500, dim))).max() * np.abs(S).max())
        c.upload_state(s, ii, jj, S)
    g = torch.Generator(device="cuda").manual_seed(1)
    x = torch.rand((n, dim + 2), dtype=torch.float64, device="cuda", generator=g)
    sid = torch.randint(-1, 3, (n,), dtype=torch.int32, device="cuda", generator=g)
    for prec in (hddm_lb.FP64, hddm_lb.F32, hddm_lb.F16X2, hddm_lb.BF16X3):
        y = torch.full((n, dofs + 3), 7.0, dtype=torch.float64, device="cuda")
        c.forward(x[:, :dim], y[:, :dofs], sid, prec)
        torch.cuda.synchronize()
        print("dim", dim, "points", n, "precision", prec, c.last_config(), flush=True)
        assert (c.last_config()["waves"] < 8) == walks
        for p0 in range(0, n, n // 5):
            m = min(3000, n - p0)
            z = torch.full((m, dofs), 7.0, dtype=torch.float64, device="cuda")
            c.forward(x[p0:p0 + m, :dim].contiguous(), z, sid[p0:p0 + m].contiguous(), prec)
            torch.cuda.synchronize()
            assert c.last_config()["waves"] >= 8
            assert (y[p0:p0 + m, :dofs] - z).abs().max() <= (1e-12 if prec == hddm_lb.FP64 else 1e-6) * most
        assert (y[:, dofs:] == 7.0).all() and (y[(sid < 0) | (sid > 1)] == 7.0).all()
    c.close()


@pytest.mark.parametrize("dim,n", [(1, 1 << 19), (2, 1 << 20), (4, 1 << 18)])
def test_adjoint_of_large_batches_in_few_dimensions(dim, n):
    """Both sides of the rule that leaves blocks that meet next to no nodes to the
    per-tile kernels: dx and dS of the default are those of formulation 1."""
    import torch
    ii, jj, lv, ix = hddm_lb.generate_grid(dim, 5, 6, 0.0, 7, 0)
    r = np.random.default_rng(dim)
    S = r.standard_normal((len(ii), 6))
    g = torch.Generator(device="cuda").manual_seed(1)
    x = torch.rand((n, dim), dtype=torch.float64, device="cuda", generator=g)
    gb = torch.randn((n, 6), dtype=torch.float64, device="cuda", generator=g)
    c = hddm_lb.Context(0)
    c.upload_state(0, ii, jj, S)
    got = []
    for form in (0, 1):
        c.set_option(hddm_lb.OPT_FORMULATION, form)
        dx, ds = torch.full_like(x, np.nan), torch.full((S.size,), np.nan, dtype=torch.float64, device="cuda")
        print("dim", dim, "points", n, "formulation", form, flush=True)
        c.adjoint(x, gb, dx, ds)
        torch.cuda.synchronize()
        got.append((dx, ds))
    c.close()
    # dS sums n terms of size B g: 1e-12 of the largest leaves room for any order
    for (a, b), tol in zip(zip(*got), (1e-10, 1e-12)):
        assert (a - b).abs().max() <= tol * b.abs().max()


@pytest.mark.parametrize("power", [99, 101, 120, -99, -101, -120])
def test_split_precision_outside_the_range_of_f32(power):
    """A dof column whose largest value lies outside 2^-100 .. 2^100 sends F16X2 to
    the walking sweeps, whose operands are scaled by column."""
    import torch
    ii, jj, lv, ix = hddm_lb.generate_grid(6, 3, 4, 0.0, 7, 0)
    r = np.random.default_rng(5)
    S = r.uniform(-1.0, 1.0, (len(ii), 5))
    S[0, 2] = 1.0
    S[:, 2] *= 2.0 ** power
    X = hddm_lb.synthetic_points(100, 6, 9)
    c = hddm_lb.Context(0)
    c.upload_state(0, ii, jj, S)
    x = torch.from_numpy(X).cuda()
    y = torch.full((100, 5), np.nan, dtype=torch.float64, device="cuda")
    print("power", power, flush=True)
    c.forward(x, y, None, hddm_lb.F16X2)
    torch.cuda.synchronize()
    assert c.last_config()["waves"] == (12 if abs(power) < 100 else 4)
    c.close()
    yo = oracle.forward(ii, jj, S, X)
    den = oracle.forward(ii, jj, np.ones((len(ii), 1)), X).max() * np.abs(S).max(axis=0)
    assert (np.abs(y.cpu().numpy() - yo).max(axis=0) <= 1e-6 * den).all()


# the second state's grid, and the waves of F32 forwards of both in one context
MIXED = [("thirds", 4), ("deep", 8), ("many hats", 8), ("fitting", 12)]


@pytest.mark.parametrize("kind,waves", MIXED, ids=lambda v: str(v))
def test_states_of_mixed_kinds_in_one_context(kind, waves):
    """What a context's sweep and adjoint are follows from all of its states."""
    import torch
    dim, dofs, n = 10, 12, 300
    r = np.random.default_rng(8)
    grids = [hddm_lb.generate_grid(dim, 2, 4, 0.3, 7, 800)[:2]]
    if kind == "thirds":
        ii, jj = (a.copy() for a in hddm_lb.generate_grid(dim, 2, 3, 0.0, 7, 0)[:2])
        third = ii == 4
        ii[third], jj[third] = 3, np.minimum(jj[third], 2)
    elif kind == "deep":
        ii = np.unique((r.random((300, dim)) < 0.8) * 2, axis=0).astype(np.int32)
        jj = ii.copy()
        assert (ii > 0).sum(1).max() >= 8
    elif kind == "many hats":
        ii, jj = hddm_lb.generate_grid(dim, 6, 7, 0.0, 7, 0)[:2]
        rows = np.sort(r.choice(len(ii), 900, replace=False))
        single = np.flatnonzero((ii > 0).sum(1) == 1)
        rows = np.unique(np.concatenate([rows, single]))
        ii, jj = np.ascontiguousarray(ii[rows]), np.ascontiguousarray(jj[rows])
    else:
        ii, jj = hddm_lb.generate_grid(dim, 2, 4, 0.3, 9, 500)[:2]
    grids.append((ii, jj))
    c = hddm_lb.Context(0)
    states = []
    for s, (i, j) in enumerate(grids):
        S = r.standard_normal((len(i), dofs))
        c.upload_state(s, i, j, S)
        states.append((i, j, S))
    X = hddm_lb.synthetic_points(n, dim, 9)
    sid = r.integers(0, 2, n).astype(np.int32)
    G = r.standard_normal((n, dofs))
    x, t, g = torch.from_numpy(X).cuda(), torch.from_numpy(sid).cuda(), torch.from_numpy(G).cuda()
    for prec, tol in ((hddm_lb.F32, 1e-6), (hddm_lb.FP64, 1e-12)):
        y = torch.full((n, dofs), np.nan, dtype=torch.float64, device="cuda")
        print(kind, "precision", prec, flush=True)
        c.forward(x, y, t, prec)
        torch.cuda.synchronize()
        if prec == hddm_lb.F32:
            assert c.last_config()["waves"] == waves
        for s, (i, j, S) in enumerate(states):
            den = oracle.forward(i, j, np.ones((len(i), 1)), X[sid == s]).max() * np.abs(S).max()
            assert np.abs(y.cpu().numpy()[sid == s] - oracle.forward(i, j, S, X[sid == s])).max() <= tol * den
    dx, ds = torch.full_like(x, np.nan), torch.full((c.surplus_offset(-1)[1],), np.nan, dtype=torch.float64, device="cuda")
    c.adjoint(x, g, dx, ds, t, hddm_lb.FP64)
    torch.cuda.synchronize()
    for s, (i, j, S) in enumerate(states):
        dxo, dso = oracle.adjoint(i, j, S, X[sid == s], G[sid == s])
        at = c.surplus_offset(s)[0]
        assert np.abs(dx.cpu().numpy()[sid == s] - dxo).max() <= 1e-10 * np.abs(dxo).max()
        assert np.abs(ds.cpu().numpy()[at:at + S.size] - dso.reshape(-1)).max() <= 1e-12 * np.abs(dso).max()
    c.close()


@pytest.mark.parametrize("case", [(6, 3, 5, 0.0, 0, 17, 17, 64), (6, 3, 5, 0.0, 0, 65, 31, 65), (16, 2, 6, 0.3, 6000, 1009, 32, 700),
                                  (17, 2, 5, 0.3, 4000, 1024, 5, 129), (32, 2, 5, 0.3, 4000, 1500, 32, 200)],
                         ids=lambda c: "d%d-n%d-c%d-p%d" % (c[0], c[5], c[6], c[7]))
def test_adjoint_of_node_subsets_against_the_oracle(case):
    """dx and dS of states whose paths have prefixes that are no nodes, at the
    edges of windows, blocks and tiles."""
    dim, base, depth, p, nodes, pick, dofs, npts = case
    r = np.random.default_rng(pick)
    ii, jj, lv, ix = hddm_lb.generate_grid(dim, base, depth, p, 7, nodes)
    rows = np.sort(r.choice(len(ii), min(pick, len(ii)), replace=False))
    ii, jj = np.ascontiguousarray(ii[rows]), np.ascontiguousarray(jj[rows])
    S, G = r.standard_normal((len(rows), dofs)), r.standard_normal((npts, dofs))
    X = hddm_lb.synthetic_points(npts, dim, 9)
    X[0] = 0.5
    c = hddm_lb.Context(0)
    c.upload_state(0, ii, jj, S)
    dx, ds = adjoint(c, X, G)
    c.close()
    dxo, dso = oracle.adjoint(ii, jj, S, X, G)
    assert np.abs(dx - dxo).max() <= 1e-10 * np.abs(dxo).max()
    assert np.abs(ds - dso.reshape(-1)).max() <= 1e-12 * np.abs(dso).max()


def test_points_far_outside_meet_no_node_of_the_direct_sweep():
    """No coordinate, however large, is inside the hat that stands for a dead
    node's: 1e300-like values, infinities and NaN give the oracle's zeros."""
    import torch
    ii, jj, lv, ix = hddm_lb.generate_grid(4, 7, 8, 0.0, 7, 0)
    S = np.random.default_rng(2).standard_normal((len(ii), 8))
    far = np.array([0x7e37e43c << 32], np.uint64).view(np.float64)[0]
    xs = [s * far / 2 ** k for k in range(9) for s in (1.0, -1.0)] + [np.inf, -np.inf, np.nan, 1e308]
    X = np.full((4 * len(xs), 4), 0.3)
    for d in range(4):
        X[d * len(xs):(d + 1) * len(xs), d] = xs
    # at these the hats of the dimension are zero, as they are just past the edge
    Y = np.where(np.abs(X) < 1.0, X, 1.5)
    yo = oracle.forward(ii, jj, S, Y)
    c = hddm_lb.Context(0)
    c.upload_state(0, ii, jj, S)
    for prec, tol in ((hddm_lb.FP64, 1e-12), (hddm_lb.F32, 1e-6)):
        for p in range(len(X)):
            x = torch.from_numpy(X[p:p + 1]).cuda()
            y = torch.zeros((1, 8), dtype=torch.float64, device="cuda")
            c.forward(x, y, None, prec)
            torch.cuda.synchronize()
            assert c.last_config()["waves"] == 8
            assert np.abs(y.cpu().numpy() - yo[p]).max() <= tol * np.abs(S).max() * 50, X[p]
    c.close()


def test_allocation_free_forward_up_to_its_limit():
    """The largest batch that five states' scratch leaves room for: 8 bytes a point,
    the histogram, cursors and 48 bytes a state in 64 MiB. One more row of 32
    points is refused."""
    import torch
    n = 8191936   # 2 (4 n + 4 * 6 * 2^15) + 256 + 256 = 2^26
    assert 2 * (4 * n + 4 * 6 * 2 ** 15) + 512 == 2 ** 26
    c = hddm_lb.Context(0)
    ii = np.array([[0], [2], [2]], np.int32)
    jj = np.array([[0], [0], [2]], np.int32)
    S = np.array([[1.0], [2.0], [4.0]])
    for s in range(5):
        c.upload_state(s, ii, jj, (s + 1) * S)
    x = torch.rand((n + 32, 1), dtype=torch.float64, device="cuda")
    sid = torch.arange(n + 32, dtype=torch.int32, device="cuda") % 5
    y = torch.full((n + 32, 1), np.nan, dtype=torch.float64, device="cuda")

    def run(m):
        return hddm_lb.lib.hddm_lb_forward_noalloc(c._h, m, x.data_ptr(), 1, sid.data_ptr(), y.data_ptr(), 1, hddm_lb.FP64, None)
    torch.cuda.synchronize()
    print("points", n, flush=True)
    assert run(n) == 0, hddm_lb.last_error()
    torch.cuda.synchronize()
    t = x[:n, 0]
    ref = (sid[:n] + 1) * (1.0 + 2.0 * (1.0 - 2.0 * t).clamp(min=0.0) + 4.0 * (2.0 * t - 1.0).clamp(min=0.0))
    assert (y[:n, 0] - ref).abs().max() <= 1e-12 * 25
    assert run(n + 32) != 0
    c.close()
