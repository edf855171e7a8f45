"""The particle push on uneven axes: a position's cell index is counted in the
axis's first spacing, so it can pass the axis by any factor.  Flat indices that
fit 32 bits, below and beyond the number of cells: the fast reduction must give
the general one's bits (spacing scaled out of the fast range by a power of
two).  Flat indices past 32 bits: every such position is past the last cell,
where the potential is zero, so particles fly straight on."""
import numpy as np
import pytest

from arbinterp_amd import workloads as W

pytestmark = pytest.mark.gpu

N = (11, 9, 14)


def _axes(rng, first):
    return [np.concatenate([[0.0, s], s + np.cumsum(rng.uniform(0.09, 0.13, size=n - 2))])
            for n, s in zip(N, first)]


def _push(axes, U, x0, v0, scale, precision, dt, steps):
    import torch
    from arbinterp_amd import ARBInterp as G
    from arbinterp_amd import batch as B
    rows = W.grid_rows(axes, [U]) * np.array([scale, scale, scale, scale * scale])
    t = G.tricubic(rows, "quiet", precision=precision)
    x, v = torch.from_numpy(x0 * scale).cuda(), torch.from_numpy(v0 * scale).cuda()
    print("push first spacing", [a[1] for a in axes], "scale", scale, precision, flush=True)
    B.push_rk4(t, x, v, dt=dt, nsteps=steps, steps_per_launch=6)
    res = x.cpu().numpy() / scale, v.cpu().numpy() / scale
    t.close()
    return res


def test_indices_within_32_bits():
    rng = np.random.default_rng(4)
    axes = _axes(rng, (0.004, 0.1, 0.02))
    lo, hi = np.array([a[1] for a in axes]), np.array([a[-2] for a in axes])
    x0 = rng.uniform(lo, hi, size=(5000, 3))
    x0[0] = hi
    x0[1::4, 0] = lo[0] + rng.uniform(0, 0.03, size=len(x0[1::4]))
    x0[1::4, 2] = lo[2] + rng.uniform(0, 0.04, size=len(x0[1::4]))
    v0 = rng.normal(scale=0.3, size=x0.shape)
    U = rng.normal(size=N)
    a = _push(axes, U, x0, v0, 1.0, "fp64", 1e-4, 13)
    b = _push(axes, U, x0, v0, 2.0 ** 310, "fp64", 1e-4, 13)
    assert not np.array_equal(a[1], v0) and np.isfinite(a[1]).any()
    for x, y in zip(a, b):
        assert np.array_equal(x, y, equal_nan=True)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("first", [(1e-9, 1e-9, 1e-9), (0.1, 0.1, 2e-9), (1e-12, 0.1, 0.1)])
def test_indices_past_32_bits(first, precision):
    rng = np.random.default_rng(6)
    axes = _axes(rng, first)
    lo, hi = np.array([a[1] for a in axes]), np.array([a[-2] for a in axes])
    x0 = rng.uniform(lo + 0.2 * (hi - lo), hi - 0.2 * (hi - lo), size=(5000, 3))
    v0 = rng.normal(scale=0.1, size=x0.shape)
    dt, steps = 1e-3, 12
    x, v = _push(axes, rng.normal(size=N), x0, v0, 1.0, precision, dt, steps)
    assert np.array_equal(v, v0)
    # straight lines: about ten roundings a step of numbers below 2
    assert np.abs(x - (x0 + steps * dt * v0)).max() < 10 * steps * 2.0 ** -53 * 2
