"""Rows with more values on an axis than the one-pass detection holds (32768):
the counts on both sides of that, rows that form no grid and would fill its
sets (refused), and a non-finite coordinate among them, wherever it stands."""
import numpy as np
import pytest

from arbinterp_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(32768, 4, 4), (4, 32769, 4), (4, 4, 150_000)])
def test_long_axes(n):
    from arbinterp_amd import ARBInterp as G
    rng = np.random.default_rng(sum(n))
    axes = [np.sort(rng.normal(size=k)) for k in n]
    rows = W.grid_rows(axes, [rng.normal(size=n)], rng)
    print("long axes", n, flush=True)
    t = G.tricubic(rows, "quiet")
    assert t._n == list(n)
    for a, x in enumerate(axes):
        assert (t._lo[a], t._hi[a], t._hh[a]) == (x[1], x[-2], abs(x[0] - x[1]))
    t.close()


@pytest.mark.parametrize("d", [3, 4])
@pytest.mark.parametrize("damage", [None, "first", "last"])
def test_no_grid(d, damage):
    from arbinterp_amd import ARBInterp as G
    rng = np.random.default_rng(3)
    rows = rng.normal(size=(1_500_000, d + 1))
    if damage:
        rows[0 if damage == "first" else -1, d - 1] = np.nan
    print("no grid", d, damage, flush=True)
    with pytest.raises(ValueError) as e:
        (G.tricubic if d == 3 else G.quadcubic)(rows, "quiet")
    assert ("non-finite" in str(e.value)) == bool(damage)
