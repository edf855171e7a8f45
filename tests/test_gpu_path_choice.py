"""Row counts on both sides of the lines between the direct and the bucketed
path: whichever the call takes by itself, the bits are those of both."""
import numpy as np
import pytest

from arbinterp_amd import _native as N
from arbinterp_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,mode,precision,least", [
    (3, "norm", "fp64", 2097152), (3, "vector", "fp64", 393216), (3, "both", "fp64", 327680),
    (3, "norm", "mixed", 1000000), (3, "vector", "mixed", 245760), (3, "both", "mixed", 286720),
    (4, "scalar", "fp64", 262144), (4, "scalar", "mixed", 800000)])
def test_either_side_of_the_line(d, mode, precision, least):
    import torch
    from arbinterp_amd import ARBInterp as G
    if d == 3:
        rows, _ = W.dipole3d(seed=5, n=(20, 18, 17), nq=1)
        t = G.tricubic(rows, "quiet", mode=mode, precision=precision)
    else:
        rows, _ = W.moving4d(seed=5, n=(9, 8, 8, 7), nq=1)
        t = G.quadcubic(rows, "quiet", precision=precision)
    q = torch.from_numpy(np.random.default_rng(3).uniform(t._lo, t._hi, size=(least + 1, d))).cuda()

    def bits(n, flags):
        out = t.query_device(q[:n], flags=flags, cells=True)
        return [x.cpu().numpy().view(np.uint8) for x in out if x is not None]

    for n in (least - 1, least):
        got = bits(n, N.ARB_Q_TIMING)
        assert (t.timings()[0] > 0) == (n >= least)     # the keys' stage: bucketed
        for flags in (N.ARB_Q_DIRECT, N.ARB_Q_SORTED):
            assert all(np.array_equal(a, b) for a, b in zip(got, bits(n, flags))), (n, flags)
    t.close()
