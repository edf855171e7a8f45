"""Fields made and dropped one after another reuse device memory: whatever a
block held before (NaN node values, another field's workspace), and whichever
thread and stream takes it, a field gives the same bits."""
import threading

import numpy as np
import pytest

from arbinterp_amd import workloads as W

pytestmark = pytest.mark.gpu


def test_threads_making_and_dropping_fields():
    import torch
    from arbinterp_amd import ARBInterp as G
    torch.cuda.synchronize()
    sizes = [(12, 11, 10), (30, 28, 26), (31, 27, 26), (18, 40, 22)]
    data, ref = [], []
    for k, n in enumerate(sizes):
        rows, q = W.dipole3d(seed=k, n=n, nq=70_000)
        t = G.tricubic(rows, "quiet", mode="both")
        ref.append([x.cpu().numpy() for x in t.query_device(torch.from_numpy(q).cuda())])
        t.close()
        bad = rows.copy()
        bad[:, 3:] = np.nan
        data.append((rows, bad, q))
    wrong = []

    def work(seed):
        rng = np.random.default_rng(seed)
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(12):
                    k = int(rng.integers(len(sizes)))
                    rows, bad, q = data[k]
                    qd = torch.from_numpy(q).cuda()
                    spoil = G.tricubic(bad, "quiet", mode="both")
                    spoil.query_device(qd)
                    del spoil                        # with its query still queued
                    t = G.tricubic(rows, "quiet", mode="both")
                    out = [x.cpu().numpy() for x in t.query_device(qd)]
                    if not all(np.array_equal(a, b) for a, b in zip(out, ref[k])):
                        wrong.append((seed, k))
                    t.close()
        except Exception as e:                       # noqa: BLE001 (reported by the test)
            wrong.append(repr(e))

    threads = [threading.Thread(target=work, args=(s,)) for s in range(3)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    assert not wrong
