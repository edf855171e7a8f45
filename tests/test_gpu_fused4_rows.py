"""The 4D kernel without a table: quads that hold no row must not run on the
position of the one they stand in for (row 0, wherever the caller has it), and
rows whose cell index passes an axis several times over (an axis whose first
spacing is its smallest) must find their cell.  The direct kernel's bits."""
import numpy as np
import pytest

from arbinterp_amd import _native as N
from arbinterp_amd import workloads as W

pytestmark = pytest.mark.gpu


def _run(t, q, flags):
    import torch
    print("rows", q.shape[0], "row 0", q[0], "flags", flags, flush=True)
    out = t.query_device(torch.from_numpy(q).cuda(), flags=flags, cells=True, out_f64=True)
    torch.cuda.synchronize()
    return [x.cpu().numpy() for x in out if x is not None]


def _same(a, b):
    return all(np.array_equal(x.view(np.uint8), y.view(np.uint8)) for x, y in zip(a, b))


@pytest.mark.parametrize("mode", ["scalar", "both"])
@pytest.mark.parametrize("first", [-3.0, 3.0, 1e6, 1e30, -1e30, np.inf, -np.inf, np.nan])
def test_row_zero_outside(first, mode):
    """Row 0 outside the box, on every axis or one, by that many spacings; one
    row inside, and partial batches of many."""
    from arbinterp_amd import ARBInterp as G
    rows, _ = W.moving4d(seed=3, n=(9, 8, 7, 6), nq=1)
    rng = np.random.default_rng(5)
    kw = {}
    if mode == "both":
        rows = np.column_stack([rows, rng.normal(size=(len(rows), 2))])
        kw = {"mode": "both"}
    t = G.quadcubic(rows, "quiet", **kw)
    lo, hi, h = np.array(t._lo), np.array(t._hi), np.array(t._hh)
    for count in (2, 700):
        for axes in ((0, 1, 2, 3), (0,), (3,)):
            q = rng.uniform(lo, hi, size=(count, 4))
            for a in axes:
                q[0, a] = (hi[a] if first > 0 else lo[a]) + first * h[a]
            ref = _run(t, q, N.ARB_Q_DIRECT)
            assert _same(ref, _run(t, q, N.ARB_Q_SORTED | N.ARB_Q_FUSED)), (count, axes)
    t.close()


def test_row_zero_outside_large_field():
    """The same where the path is taken by itself (a table of about 300 MB)."""
    from arbinterp_amd import ARBInterp as G
    rows, _ = W.moving4d(seed=4, n=(22, 21, 20, 27), nq=1)
    t = G.quadcubic(rows, "quiet")
    q = np.random.default_rng(2).uniform(t._lo, t._hi, size=(300_001, 4))
    q[0] = 1e30
    q[1:4, 2] = (-1e30, np.inf, np.nan)
    got = _run(t, q, 0)
    assert t.field_info().table_built == 0
    assert _same(_run(t, q, N.ARB_Q_TABLE | N.ARB_Q_DIRECT), got)
    t.close()


def test_rows_past_an_uneven_axis():
    """Axes of 8 x 9 x 10 x 6 nodes, the first spacing along x and z a fraction
    of the others: indices along x of up to 170 for its 5 cells, along z of up
    to 37 for its 7, flat indices below and beyond the number of cells."""
    from arbinterp_amd import ARBInterp as G
    rng = np.random.default_rng(7)
    axes = [np.concatenate([[0.0, s], s + np.cumsum(rng.uniform(0.8, 1.2, size=n - 2))])
            for n, s in ((8, 0.03), (9, 1.0), (10, 0.2), (6, 0.9))]
    vals = rng.normal(size=(8, 9, 10, 6))
    t = G.quadcubic(W.grid_rows(axes, [vals], rng), "quiet")
    lo, hi = np.array(t._lo), np.array(t._hi)
    q = rng.uniform(lo, hi, size=(4000, 4))
    q[::3, 3] = lo[3] + (q[::3, 3] - lo[3]) * 0.2
    ref = _run(t, q, N.ARB_Q_DIRECT)
    past = np.floor((q[:, 0] - lo[0]) / t._hh[0]) >= 5
    inside = ref[-1] < t.field_info().nc
    assert (past & inside).sum() > 300 and (past & ~inside).sum() > 300
    assert _same(ref, _run(t, q, N.ARB_Q_SORTED | N.ARB_Q_FUSED))
    t.close()
