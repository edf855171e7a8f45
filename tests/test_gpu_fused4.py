"""The 4D kernel that forms coefficients from node values, four lanes to a row:
the direct kernel's bits (the table) where it can go wrong, and the calls that
take it by themselves."""
import numpy as np
import pytest

from arbinterp_amd import _native as N
from arbinterp_amd import workloads as W

pytestmark = pytest.mark.gpu


def _run(t, q, flags):
    import torch
    out = t.query_device(torch.from_numpy(q).cuda(), flags=flags, cells=True, out_f64=True)
    torch.cuda.synchronize()
    return [x.cpu().numpy() for x in out if x is not None]


def _same(a, b, tag):
    for x, y in zip(a, b):
        assert np.array_equal(x.view(np.uint8), y.view(np.uint8)), tag


def _rows(n, ncomp, nan_node=None):
    rows, _ = W.moving4d(seed=3, n=n, nq=1)
    rng = np.random.default_rng(8)
    cols = [rows[:, 4]] + [rng.normal(size=len(rows)) for _ in range(ncomp - 1)]
    rows = np.column_stack([rows[:, :4]] + cols)
    if nan_node is not None:
        at = np.all([rows[:, a] == np.unique(rows[:, a])[nan_node[a]] for a in range(4)], axis=0)
        rows[at, 4] = np.nan
    return rows


@pytest.mark.parametrize("mode,precision", [("scalar", "fp64"), ("vector", "fp64"),
                                            ("norm", "mixed"), ("both", "fp64")])
@pytest.mark.parametrize("n", [(4, 4, 4, 4), (7, 7, 5, 5), (8, 9, 10, 6), (5, 6, 5, 70)])
def test_blocks_layers_and_batches(n, mode, precision):
    """One cell; one full block; remainders on every axis; more layers of t
    than one workgroup takes.  From one row to more than a workgroup's chunk in
    a block (several batches of 64, shared buckets), rows in one cell, layers
    without rows between others; coordinates on IntMin and IntMax (aliased
    cells), a NaN node."""
    from arbinterp_amd import ARBInterp as G
    nan_node = tuple(k - 2 for k in n) if n[3] == 6 else None
    rows = _rows(n, 1 if mode == "scalar" else 3, nan_node)
    kw = {} if mode == "scalar" else {"mode": mode}
    t = G.quadcubic(rows, "quiet", precision=precision, **kw)
    rng = np.random.default_rng(1)
    for count in (1, 63, 130, 1100, 9000):
        q = rng.uniform(t._lo, t._hi, size=(count, 4))
        if count >= 1100:
            q[:, 3] = np.where(rng.random(count) < 0.7, q[0, 3], q[:, 3])
        q[::97, 0] = t._hi[0]
        q[::89, 2] = t._lo[2]
        q[::83, 3] = t._hi[3]
        if count == 1100:
            q[:] = np.minimum(q[-1] + rng.uniform(0, 1e-3, size=q.shape) * t._hh, t._hi)
        # a coordinate at IntMax may reduce past the sentinel: clamped by both
        ref = _run(t, q, N.ARB_Q_DIRECT)
        got = _run(t, q, N.ARB_Q_SORTED | N.ARB_Q_FUSED)
        _same(ref, got, (n, mode, precision, count))
        import torch
        qd = torch.from_numpy(q).cuda()
        a = t.query_packed(qd, flags=N.ARB_Q_DIRECT).cpu().numpy()
        b = t.query_packed(qd, flags=N.ARB_Q_SORTED | N.ARB_Q_FUSED).cpu().numpy()
        _same([a], [b], (n, mode, precision, count, "packed"))
    t.close()


@pytest.mark.parametrize("d", [3, 4])
def test_large_field_without_a_table(d):
    """A field whose table (about 300 MB) exceeds the Infinity Cache is queried
    without one by itself, then allocation-free with the same results; the
    table's bits."""
    import ctypes
    import torch
    from arbinterp_amd import ARBInterp as G
    if d == 3:
        rows, q = W.dipole3d(seed=4, n=(90, 60, 37), nq=200_003)
        t = G.tricubic(rows, "quiet", mode="both")
    else:
        rows, _ = W.moving4d(seed=4, n=(22, 21, 20, 27), nq=1)
        t = G.quadcubic(rows, "quiet")
        q = np.random.default_rng(2).uniform(t._lo, t._hi, size=(300_001, 4))
    assert t.field_info().table_bytes > 256 << 20
    got = _run(t, q, 0)
    assert t.field_info().table_built == 0
    qd = torch.from_numpy(q).cuda()
    out = [torch.empty_like(x) for x in t.query_device(qd) if x is not None]
    ptr = [ctypes.c_void_p(x.data_ptr()) for x in out]
    if d == 4:
        ptr = [None] + ptr
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for n in (len(q), 1000):
        N.check(N.lib().arb_query_noalloc(t._h, ctypes.c_void_p(qd.data_ptr()), n, d, *ptr, None,
                                          0, s), "noalloc")
        torch.cuda.synchronize()
        for x, y in zip(out, got):
            assert np.array_equal(x[:n].cpu().numpy().view(np.uint8), y[:n].view(np.uint8))
    assert t.field_info().table_built == 0
    _same(_run(t, q, N.ARB_Q_TABLE | N.ARB_Q_SORTED), got, "table")
    _same(_run(t, q, 0), got, "with a table")
    t.close()
