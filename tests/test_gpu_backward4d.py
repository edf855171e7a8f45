"""4D node adjoint at the edges of its blocks (4 x 4 x 2 cells in x, y, z, all
of t): one cell per axis, blocks with a remainder on every axis, layers of t
without queries before, between and after those with some.  Against the
oracle's FP64 adjoint: both are FP64 sums of the same terms (at most 256
entries of order one times a few hundred queries a node), so they agree to
some 1e3 roundings of the largest component, 1e-12; the bound is 1e-11."""
import numpy as np
import pytest

from arbinterp_amd import workloads as W
from oracle import arbinterp_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,layers", [
    ((4, 4, 4, 4), (0,)),                    # one cell
    ((7, 7, 5, 5), (0, 1)),                  # one full block
    ((8, 8, 6, 4), (0,)),                    # one cell past a block on x, y, z
    ((10, 9, 8, 14), (1, 2, 9)),             # gaps of t: more than the four planes a cell touches
    ((9, 12, 7, 16), tuple(range(13))),
])
def test_backward_4d_block_edges(n, layers):
    import torch
    from arbinterp_amd import ARBInterp as G
    from arbinterp_amd import autograd as AG
    rows, _ = W.moving4d(seed=3, n=n, nq=1)
    t = G.quadcubic(rows.copy(), "quiet")
    lo, hi = np.array(t._lo), np.array(t._hi)
    rng = np.random.default_rng(sum(n))
    q = rng.uniform(lo, hi, size=(400, 4))
    q[:, 3] = lo[3] + t.ht * (rng.choice(layers, size=400) + rng.uniform(0.05, 0.95, size=400))
    w = rng.normal(size=400)
    fld = AG.DifferentiableField(t, dtype=torch.float64)
    x = torch.from_numpy(q).cuda().requires_grad_(True)
    U, g = fld(x)
    ((torch.from_numpy(w).cuda() * U).sum() + (g * g).sum()).backward()
    o = O.quadcubic(rows.copy(), "quiet")
    _, og = o.Query(q.copy())
    _, ref = o.backward(q, w, 2 * og)
    got = fld.values.grad.cpu().numpy()
    assert np.abs(got - ref).max() <= 1e-11 * np.abs(ref).max()
    t.close()
