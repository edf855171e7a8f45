"""Detection of the grid's axes in one pass: axes longer than the values that
come back with the first copy (1024) and than the pass holds (32768: hash sets
for any rows), negative zeros, rows in any order, and the grids that are
refused, against numpy's unique values."""
import numpy as np
import pytest

from arbinterp_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(4, 5, 6), (1500, 4, 5), (4, 4, 3000), (40000, 4, 4), (7, 6, 5, 4),
                               (4, 4, 4, 1100)])
@pytest.mark.parametrize("even", [True, False])
def test_axes_and_node_order(n, even):
    import torch
    from arbinterp_amd import ARBInterp as G
    from arbinterp_amd.autograd import node_values
    rng = np.random.default_rng(sum(n))
    axes = [np.arange(k) * 0.25 - 1.0 if even else np.sort(rng.normal(size=k)) for k in n]
    vals = rng.normal(size=n)
    rows = W.grid_rows(axes, [vals], rng)
    if even:
        z = rows[:, 0] == 0.0
        rows[z, 0] = np.where(rng.random(z.sum()) < 0.5, -0.0, 0.0)
    t = (G.tricubic if len(n) == 3 else G.quadcubic)(rows, "quiet")
    assert t._n == list(n)
    for a, x in enumerate(axes):
        assert (t._lo[a], t._hi[a], t._hh[a]) == (x[1], x[-2], abs(x[0] - x[1]))
    got = node_values(t).cpu().numpy()[0]
    assert np.array_equal(got, vals.transpose(*reversed(range(len(n)))).reshape(-1))
    t.close()
    torch.cuda.empty_cache()


@pytest.mark.parametrize("damage", ["duplicate", "missing", "nan", "inf", "scattered"])
def test_refused_rows(damage):
    from arbinterp_amd import ARBInterp as G
    rng = np.random.default_rng(2)
    rows = W.grid_rows([np.arange(k) * 0.5 for k in (9, 8, 7)], [rng.normal(size=(9, 8, 7))], rng)
    if damage == "duplicate":
        rows[17, :3] = rows[400, :3]
    elif damage == "missing":
        rows = rows[:-1]
    elif damage == "nan":
        rows[3, 1] = np.nan
    elif damage == "inf":
        rows[503, 2] = -np.inf
    else:
        rows = rng.normal(size=(50_000, 4))
    with pytest.raises(ValueError):
        G.tricubic(rows, "quiet")
