"""lscomp_release_all while other threads are in calls: their scratch areas live
until those calls have ended, so every result stays right."""
import threading

import numpy as np
import pytest

from lsc_helpers import MODES, synth

pytestmark = pytest.mark.gpu


def test_release_during_calls(gpu, orc):
    import torch
    shape = (8, 200, 300)
    a = synth("cssi", shape, seed=3)
    b = (a // 5 * 5).astype(np.uint16)
    bins, p = MODES["lossless"]
    _, ref, refn = orc.compress(a, bins, p)
    want = orc.ssim(a, b)
    sq = int(((a.astype(np.int64) - b) ** 2).sum())
    da, db = (torch.from_numpy(v.view(np.int16)).cuda() for v in (a, b))
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(3)]
    wrong = []

    def work(stream):
        try:
            torch.cuda.set_device(0)
            with torch.cuda.stream(stream):
                for _ in range(60):
                    if gpu.error_stats(da, db)["sum_sq_err"] != sq:
                        wrong.append("error_stats")
                    if abs(gpu.ssim(da, db, shape) - want) > 1e-10:
                        wrong.append("ssim")
                    out, n = gpu.compress(da, shape, bins, p)
                    if n != refn or not np.array_equal(out[:n].cpu().numpy(), ref):
                        wrong.append("compress")
        except Exception as e:   # reported by the test, not lost in the thread
            wrong.append(repr(e))

    threads = [threading.Thread(target=work, args=(s,)) for s in streams]
    for t in threads:
        t.start()
    while any(t.is_alive() for t in threads):
        gpu.release_all()
    for t in threads:
        t.join()
    assert wrong == []
