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
