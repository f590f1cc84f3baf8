"""Contexts of several host threads whose kernels are the same and whose LDS tables are not: each
thread creates its context and runs two subints while the others do, and every result equals the one
of the same job alone, bit for bit."""
import threading

import numpy as np
import pytest

from difx_amd import config as cf
from difx_amd.core import FxCore
from fxcases import slot

pytestmark = pytest.mark.gpu
OFFS = (0, 1, 0)


def _job(stride, order):
    cfg = cf.standard_config(2, 1, [4800.0], 32.0, 8192, subint_ns=5 * 256000, xengine="fp16", seed=99,
                             fringe_rot_order=order, max_delay_us=50.0)
    for d in cfg.datastreams:
        d.arraystridelen = stride
    return cfg


def test_threads_with_tables_of_different_sizes(gpu):
    jobs = [_job(s, o) for o in (1, 2) for s in (64, 128, 256)]
    data = [slot(c, OFFS, seed=100) for c in jobs]
    alone = []
    for c, (d, k) in zip(jobs, data):
        with FxCore(c) as core:
            alone.append(core.processdata(OFFS, d, k))
    got = [[] for _ in jobs]

    def work(i):
        with FxCore(jobs[i]) as core:
            for _ in range(2):
                got[i].append(core.processdata(OFFS, *data[i]))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(jobs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for i in range(len(jobs)):
        assert len(got[i]) == 2
        for g in got[i]:
            np.testing.assert_array_equal(g.view(np.uint64), alone[i].view(np.uint64))
