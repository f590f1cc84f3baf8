"""The X-engines' loop over FFTs in several parts, and the accumulation in several batches of freqs, against the FP64 oracle: a subint in ten parts,
in three chunks of which the last is short, in two of which the last has fewer steps than parts
(parts of it stay empty), and two tiles of rows.  The number of parts is read from the tables
first: a case that no longer splits fails.  Batches: averaged products against the averages of the
same job's unaveraged ones, which need no accumulator (to FP32 rounding of four terms, 3e-7).  Bars: the parity bars of the FP32 (1e-5), FP16 (1e-3)
and BF16 (1e-2) visibilities per record."""
import numpy as np
import pytest

import fxoracle as fo
from difx_amd import config as cf
from fxcases import record_errors, slot
from test_x_targets_cpu import extents

pytestmark = pytest.mark.gpu
BAR = {"fp32": 1e-5, "fp16": 1e-3, "bf16": 1e-2}
OFFS = (0, 1, 0)


@pytest.mark.parametrize("xe", ["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("rows,ffts,chunk", [(8, 700, 0), (8, 700, 264), (8, 648, 640), (33, 260, 0), (40, 264, 256)])
def test_parts(gpu, xe, rows, ffts, chunk):
    from difx_amd.core import FxCore
    npol = 2 if rows % 2 == 0 else 1
    cfg = cf.standard_config(rows // npol, npol, [4800.0], 16.0, 128, subint_ns=ffts * 8000, xengine=xe, seed=71,
                             chunk_ffts=chunk, max_delay_us=50.0)
    *_, run, parts, _ = extents(cfg)
    assert parts >= min(run, chunk or run) // 64 > 1
    data, ctrl = slot(cfg, OFFS, seed=72)
    ref, _ = fo.process_subint(cfg, list(OFFS), data, ctrl)
    lay = fo.result_layout(cfg)
    with FxCore(cfg) as core:
        first = core.processdata(OFFS, data, ctrl)
        again = core.processdata(OFFS, data, ctrl)
    np.testing.assert_array_equal(first.view(np.uint64), again.view(np.uint64))
    e = record_errors(cfg, lay, first.astype(np.complex128), ref)
    print(xe, parts, "parts,", len(e["cross"]), "records, max", max(e["cross"]), "auto", max(e["auto"]), flush=True)
    assert max(e["cross"]) < BAR[xe] and max(e["auto"]) < BAR[xe]


@pytest.mark.parametrize("xe", ["fp32", "fp16"])
def test_batches(gpu, xe):
    """4 freqs of 32 rows x 8192 channels averaged by 4: 138 MB of products, in several batches."""
    from difx_amd.core import FxCore

    def job(avg):
        cfg = cf.standard_config(16, 2, [4800.0 + 40.0 * k for k in range(4)], 32.0, 8192, subint_ns=8 * 256000,
                                 xengine=xe, seed=73, max_delay_us=50.0)
        for f in cfg.freqs:
            f.chanavg = avg
        return cfg

    cfg = job(4)
    assert extents(cfg)[8] > 1
    data, ctrl = slot(cfg, OFFS, seed=74)
    with FxCore(job(1)) as core:
        whole = core.processdata(OFFS, data, ctrl)
    with FxCore(cfg) as core:
        got = core.processdata(OFFS, data, ctrl)
    la, lw = fo.result_layout(cfg), fo.result_layout(job(1))
    spans = [(la.baseline_off[k], lw.baseline_off[k], 4) for k in la.baseline_off]
    spans += [(la.autocorr_off[d], lw.autocorr_off[d], 16) for d in range(16)]
    for a, w, n in spans:
        want = whole[w: w + n * 8192].reshape(-1, 4).astype(np.complex128).mean(axis=1)
        assert np.max(np.abs(got[a: a + n * 2048] - want)) <= 3e-7 * np.max(np.abs(whole[w: w + n * 8192]))
