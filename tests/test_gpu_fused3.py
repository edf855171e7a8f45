"""The 3D kernel that forms coefficients in registers, two rows of a cell per
lane: the direct kernel's bits (the table) where it can go wrong."""
import numpy as np
import pytest

from arbinterp_amd import _native as N
from arbinterp_amd import workloads as W

pytestmark = pytest.mark.gpu


def _run(t, q, flags):
    import torch
    out = t.query_device(torch.from_numpy(q).cuda(), flags=flags, cells=True)
    torch.cuda.synchronize()
    return [x.cpu().numpy() for x in out if x is not None]


def _same(a, b, tag):
    for x, y in zip(a, b):
        assert np.array_equal(x.view(np.uint8), y.view(np.uint8)), tag


@pytest.mark.parametrize("n", [(7, 7, 7), (8, 9, 10), (19, 6, 13)])
@pytest.mark.parametrize("mode,precision", [("scalar", "fp64"), ("vector", "fp64"),
                                            ("both", "fp64"), ("both", "mixed")])
def test_rows_per_cell_and_rounds(n, mode, precision):
    """From one row in all to several hundred per 4 x 4 x 4 block: cells with
    odd and even numbers of rows, more pairs than threads (a second round: 64
    cells, some 500 rows), more rows than a workgroup takes (shared buckets),
    rows in one cell; coordinates on IntMin, IntMax (an aliased cell) and in
    the last cells of edge blocks."""
    from arbinterp_amd import ARBInterp as G
    rows, _ = W.dipole3d(seed=3, n=n, nq=1)
    if mode == "scalar":
        rows = rows[:, :4]
    kw = {} if mode == "scalar" else {"mode": mode}
    t = G.tricubic(rows, "quiet", precision=precision, **kw)
    rng = np.random.default_rng(1)
    blocks = np.prod([-(-(k - 3) // 4) for k in n])
    for count in (1, 2, 129, 505 * blocks, 2100 * blocks):
        q = rng.uniform(t._lo, t._hi, size=(int(count), 3))
        q[::97, 0] = t._hi[0]
        q[::89, 2] = t._lo[2]
        if count == 129:
            q[:] = q[-1] + rng.uniform(0, 1e-3, size=q.shape) * t._hh
            q = np.minimum(q, t._hi)
        # a coordinate at IntMax may reduce past the sentinel: clamped by both
        ref = _run(t, q, N.ARB_Q_DIRECT | N.ARB_Q_TABLE)
        got = _run(t, q, N.ARB_Q_SORTED | N.ARB_Q_FUSED)
        _same(ref, got, (n, mode, precision, count))
    t.close()


def test_large_fp64_field_takes_it_by_size():
    """A 'vector' field whose table (427 MB) exceeds the Infinity Cache is
    queried without one, bit for bit as with it; the table is built when
    asked for."""
    from arbinterp_amd import ARBInterp as G
    rows, q = W.dipole3d(seed=4, n=(100, 64, 50), nq=200_003)
    t = G.tricubic(rows, "quiet", mode="vector")
    got = _run(t, q, 0)
    assert t.field_info().table_built == 0
    _same(_run(t, q, N.ARB_Q_TABLE), got, "auto")
    assert t.field_info().table_built == 1
    _same(_run(t, q, 0), got, "with a table")
    t.close()
