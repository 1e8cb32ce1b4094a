"""States that hold a node more than once, the root among them: every copy is a
node of its own, as the oracle's sum over nodes has it."""
import numpy as np
import pytest

import hddm_lb
import oracle
from test_host import walk_layout, walk_layout_static


def state(dim=5, dofs=6, seed=3):
    ii, jj, lv, ix = hddm_lb.generate_grid(dim, 3, 4, 0.0, 1, 0)
    r = np.random.default_rng(seed)
    # copies of 150 nodes, some of them several, three of the root
    again = np.concatenate([r.integers(0, len(ii), 150), np.flatnonzero(~(ii | jj).any(1)).repeat(3)])
    ii, jj = np.concatenate([ii, ii[again]]), np.concatenate([jj, jj[again]])
    mix = r.permutation(len(ii))
    return np.ascontiguousarray(ii[mix]), np.ascontiguousarray(jj[mix]), r.standard_normal((len(ii), dofs)), r


def test_host_layout_has_an_op_for_every_copy():
    ii, jj, S, r = state()
    L = hddm_lb.Layout(ii, jj, S)
    assert sorted(L.op_node[L.op_last]) == list(range(L.nno))
    assert (L.skip > np.arange(L.nops)).all() and (L.skip <= L.nops).all()
    assert (L.op_relskip == L.skip - np.arange(L.nops)).all()
    X = r.random((64, ii.shape[1]))
    yo = oracle.forward(ii, jj, S, X)
    for walk in (walk_layout, walk_layout_static):
        y = walk(L, X, S[L.order])[0]
        # sums of some 300 terms in another order
        assert np.abs(y - yo).max() <= 1e-12 * np.abs(yo).max()


@pytest.mark.gpu
@pytest.mark.parametrize("form", [0, 1, 2])
def test_forward_and_adjoint_with_copies(form):
    import torch
    ii, jj, S, r = state()
    X, G = r.random((200, ii.shape[1])), r.standard_normal((200, S.shape[1]))
    yo, (dxo, dso) = oracle.forward(ii, jj, S, X), oracle.adjoint(ii, jj, S, X, G)
    ctxs = []
    for device in (1, 0):
        c = hddm_lb.Context(0)
        c.set_option(hddm_lb.OPT_DEVICE_LAYOUT, device)
        c.upload_state(0, ii, jj, S)
        c.set_option(hddm_lb.OPT_FORMULATION, form)
        ctxs.append(c)
    for name in hddm_lb.STATE_ARRAYS:
        assert np.array_equal(ctxs[0].state_array(0, name), ctxs[1].state_array(0, name)), name
    x, g = torch.from_numpy(X).cuda(), torch.from_numpy(G).cuda()
    for c in ctxs:
        for prec, tol in ((hddm_lb.FP64, 1e-12), (hddm_lb.F32, 1e-6), (hddm_lb.F16X2, 1e-6)):
            print("formulation", form, "precision", prec, flush=True)
            y = torch.full((200, S.shape[1]), np.nan, dtype=torch.float64, device="cuda")
            c.forward(x, y, None, prec)
            torch.cuda.synchronize()
            assert np.abs(y.cpu().numpy() - yo).max() <= tol * np.abs(yo).max()
        dx, ds = torch.full_like(x, np.nan), torch.full((S.size,), np.nan, dtype=torch.float64, device="cuda")
        c.adjoint(x, g, dx, ds, None, hddm_lb.FP64)
        torch.cuda.synchronize()
        assert np.abs(dx.cpu().numpy() - dxo).max() <= 1e-10 * np.abs(dxo).max()
        assert np.abs(ds.cpu().numpy() - dso.reshape(-1)).max() <= 1e-12 * np.abs(dso).max()
        c.close()
