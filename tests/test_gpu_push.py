"""The push's fast reduction and division against the general ones.

Scaling positions, velocities and spacing by s = 2^310 and the potential by
s^2 scales every operation of the push exactly (powers of two, far from
overflow), while the spacing leaves the range of the fast division: the
general path must give the fast one's trajectories times s, bit for bit.
Particles start in every cell of an odd-sized grid, some beside the faces
(and leave the box), one exactly on the upper corner."""
import numpy as np
import pytest

from arbinterp_amd import workloads as W

pytestmark = pytest.mark.gpu


def test_fast_push_equals_general():
    import torch
    from arbinterp_amd import ARBInterp as G
    from arbinterp_amd import batch as B
    n, h = (11, 9, 14), (0.1, 0.13, 0.07)
    rng = np.random.default_rng(3)
    axes = W.grid_axes(n, h)
    U = rng.normal(size=n)
    rows = W.grid_rows(axes, [U], rng)
    lo = np.array([a[1] for a in axes])
    hi = np.array([a[-2] for a in axes])
    x0 = rng.uniform(lo, hi, size=(5000, 3))
    x0[0] = hi
    x0[1:4] = lo + 1e-6
    v0 = rng.normal(scale=0.3, size=x0.shape)
    s = 2.0 ** 310
    res = []
    for scale in (1.0, s):
        r = rows * np.array([scale, scale, scale, scale * scale])
        t = G.tricubic(r, "quiet")
        x = torch.from_numpy(x0 * scale).cuda()
        v = torch.from_numpy(v0 * scale).cuda()
        B.push_rk4(t, x, v, dt=1e-2, nsteps=25, steps_per_launch=6)
        res.append((x.cpu().numpy() / scale, v.cpu().numpy() / scale))
        t.close()
    assert np.isnan(res[0][0]).any() and not np.isnan(res[0][0]).all()
    for a, b in zip(*res):
        assert np.array_equal(a, b, equal_nan=True)
