"""Node adjoint of cells that hold about a chunk of queries (3D 256, 4D 128):
one fewer, as many, one more, two chunks and one more, in neighbouring cells so
that chunks start inside them at any place.  Against the oracle's FP64 adjoint:
sums of at most some thousand terms of the same size in another order, 1e-12 of
the largest component; the bound is 1e-11."""
import numpy as np
import pytest

from arbinterp_amd import workloads as W
from oracle import arbinterp_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,chunk", [(3, 256), (4, 128)])
def test_backward_chunk_edges(d, chunk):
    import torch
    from arbinterp_amd import ARBInterp as G
    from arbinterp_amd import autograd as AG
    n = (9, 8, 7) if d == 3 else (8, 7, 7, 6)
    rows, _ = W.moving4d(seed=3, n=n if d == 4 else n + (4,), nq=1)
    if d == 3:
        rows = rows[rows[:, 3] == rows[0, 3]][:, [0, 1, 2, 4]]
    cls, ocls = (G.tricubic, O.tricubic) if d == 3 else (G.quadcubic, O.quadcubic)
    t = cls(rows.copy(), "quiet")
    rng = np.random.default_rng(d)
    q = []
    for k, count in enumerate((3, chunk - 1, chunk, chunk + 1, 2 * chunk + 1, 5)):
        cell = np.array([k % (n[0] - 3), k // (n[0] - 3)] + [1] * (d - 2))
        q.append(t._lo + (cell + rng.uniform(0.05, 0.95, size=(count, d))) * t._hh)
    q = np.concatenate(q)
    q = q[rng.permutation(len(q))]
    w = rng.normal(size=len(q))
    fld = AG.DifferentiableField(t, dtype=torch.float64)
    x = torch.from_numpy(q).cuda().requires_grad_(True)
    U, g = fld(x)
    ((torch.from_numpy(w).cuda() * U).sum() + (g * g).sum()).backward()
    o = ocls(rows.copy(), "quiet")
    _, og = o.Query(q.copy())
    _, ref = o.backward(q, w, 2 * og)
    got = fld.values.grad.cpu().numpy()
    assert np.abs(got - ref).max() <= 1e-11 * np.abs(ref).max()
    t.close()
