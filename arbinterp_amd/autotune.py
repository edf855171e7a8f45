"""Autotuner for the query kernels.

`tune_query(interp, q)` times the candidate launch shapes of one interpolator
on the caller's own positions (GPU, HIP events on the current stream):

  * the direct lane-per-query kernel;
  * the cell-bucketed kernel staging coefficients from the table
    (ARB_Q_TABLE) and the default bucketed kernel, for every block of cells
    (cells per axis) on a ladder whose LDS footprint fits, with 64/128/256
    threads per workgroup; and the bucketed path as the library chooses it.

Outputs that must not depend on the launch shape are compared bit for bit:
every table-staged candidate against the first one, and the default
candidates of one block against each other.  Where the default kernels are
the node-tile ones (mixed precision, 3D), their FP32 rounding depends on
the block (each block has its own tile models) and differs from the
table's, so across blocks and families the outputs are compared with the
direct kernel's within a tolerance (`_close`).  A failed comparison
raises.  The fastest
candidate is applied (`interp.set_tuning`, `interp.default_flags`) and
remembered per (grid, mode, precision, query-count octave) for the process.

`tune_batch(batch, q, counts)` does the same for the batched launch (queries
per work item, threads per workgroup, workgroups per compute unit).
"""
from __future__ import annotations

import itertools
import math

import torch

from . import _native as N

_CACHE: dict = {}


def _key(interp, n):
    info = interp._info
    return (interp.NDIM, tuple(int(info.n[a]) for a in range(interp.NDIM)), int(info.mode),
            int(info.precision), int(math.log2(max(1, n))))


def block_ladder(interp, max_lds=64 * 1024):
    """Candidate cell blocks (one edge per axis) whose LDS stage fits."""
    d = interp.NDIM
    K = 4 ** d
    esz = 8 if interp.precision == "fp64" else 4
    cellbytes = (interp._info.ninterp * K * esz // 16 + 1) * 16
    edges = (1, 2, 4, 8)
    out = []
    for b in itertools.product(edges, repeat=d):
        cells = math.prod(b)
        if cells * cellbytes > max_lds or cells > 128:
            continue
        if any(b[a] > int(interp._info.npos[a]) for a in range(d)):
            continue
        out.append(b)
    return out


def _same(a, b):
    for x, y in zip(a, b):
        if x is None and y is None:
            continue
        if not torch.equal(torch.nan_to_num(x, nan=1e300), torch.nan_to_num(y, nan=1e300)):
            return False
    return True


def _close(a, b, rtol=1e-5, floor=1e-3):
    """Same NaN pattern, and |x - y| <= rtol (|y| + floor max|y|) elementwise
    per output (the floor covers components that cross zero)."""
    for x, y in zip(a, b):
        if x is None and y is None:
            continue
        if x.dtype == torch.int64:
            if not torch.equal(x, y):
                return False
            continue
        x64, y64 = x.double(), y.double()
        nx, ny = torch.isnan(x64), torch.isnan(y64)
        if not torch.equal(nx, ny):
            return False
        x64, y64 = x64[~nx], y64[~ny]
        if y64.numel() == 0:
            continue
        tol = rtol * (y64.abs() + floor * float(y64.abs().max()))
        if not bool(((x64 - y64).abs() <= tol).all()):
            return False
    return True


def _time(fn, reps):
    fn()
    torch.cuda.synchronize()
    e0 = torch.cuda.Event(enable_timing=True)
    e1 = torch.cuda.Event(enable_timing=True)
    e0.record()
    for _ in range(reps):
        fn()
    e1.record()
    torch.cuda.synchronize()
    return e0.elapsed_time(e1) / reps


def tune_query(interp, q, reps=3, max_candidates=None, verify=True, use_cache=True):
    """Pick the fastest launch shape for queries like `q` (CUDA float64 tensor).
    Returns {"path" ("direct", "table" or "sorted"), "block", "threads", "ms",
    "table": [(cand, ms), ...]}."""
    n = q.shape[0]
    key = _key(interp, n)
    if use_cache and key in _CACHE:
        best = _CACHE[key]
        _apply(interp, best)
        return dict(best, cached=True)
    out = interp.query_device(q, flags=N.ARB_Q_DIRECT)
    ref = tuple(t.clone() if t is not None else None for t in out)
    cands = [("direct", None, 0), ("sorted", None, 0)]
    for b in block_ladder(interp):
        for th in (64, 128, 256):
            cands.append(("table", b, th))
            cands.append(("sorted", b, th))
    if max_candidates:
        cands = cands[:max_candidates]
    table = []
    first = {}        # "table" / block -> outputs of its first candidate
    for path, b, th in cands:
        if path == "direct":
            interp.set_tuning(None, 0)
            fl = N.ARB_Q_DIRECT
        else:
            interp.set_tuning(b, th)
            fl = N.ARB_Q_SORTED | (N.ARB_Q_TABLE if path == "table" else 0)
        fn = lambda: interp.query_device(q, flags=fl, out=out)
        ms = _time(fn, reps)
        if verify:
            key = "table" if path == "table" else b
            if path == "direct":
                ok = _same(out, ref)
            elif key in first:
                ok = _same(out, first[key])
            else:
                ok = _close(out, ref)
                first[key] = tuple(t.clone() if t is not None else None for t in out)
            if not ok:
                raise RuntimeError("autotune: launch shape %s %s %d changed the results"
                                   % (path, b, th))
        table.append(((path, b, th), ms))
    (path, b, th), ms = min(table, key=lambda x: x[1])
    best = {"path": path, "block": b, "threads": th, "ms": ms}
    _apply(interp, best)
    _CACHE[key] = best
    return dict(best, table=table, cached=False)


def _apply(interp, best):
    if best["path"] == "direct":
        interp.set_tuning(None, 0)
        interp.default_flags = N.ARB_Q_DIRECT
    else:
        interp.set_tuning(best["block"], best["threads"])
        interp.default_flags = N.ARB_Q_SORTED | (N.ARB_Q_TABLE if best["path"] == "table" else 0)


def tune_batch(batch, q, counts, reps=3, verify=True):
    """Pick (chunk, threads, blocks_per_cu) for a FieldBatch and these counts."""
    ref = tuple(t.clone() if t is not None else None for t in batch.query(q, counts))
    out = batch.query(q, counts)
    table = []
    for chunk, th, bpc in itertools.product((64, 128, 256, 512, 1024), (64, 128, 256), (2, 4, 8)):
        if th > chunk:
            continue
        batch.set_tuning(chunk, th, bpc)
        ms = _time(lambda: batch.query(q, counts, out=out), reps)
        if verify and not _same(out, ref):
            raise RuntimeError("autotune: batch shape (%d,%d,%d) changed the results" % (chunk, th, bpc))
        table.append(((chunk, th, bpc), ms))
    (chunk, th, bpc), ms = min(table, key=lambda x: x[1])
    batch.set_tuning(chunk, th, bpc)
    return {"chunk": chunk, "threads": th, "blocks_per_cu": bpc, "ms": ms, "table": table}
