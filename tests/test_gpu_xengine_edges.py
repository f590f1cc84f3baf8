"""The X-engines at the edges of their row classes and FFT ranges, against the FP64 oracle: row
counts around the 16-, 32- and 64-row tiles, FFT counts that leave split ranges and stages
short, and zoom windows of
odd width and offset (a last channel on its own, rows that are not 16-byte aligned).  Bars: the
parity bars of the FP32 (1e-5) and FP16 (1e-3) visibilities per record."""
import numpy as np
import pytest

import fxoracle as fo
from difx_amd import config as cf
from fxcases import record_errors, slot

pytestmark = pytest.mark.gpu
BAR = {"fp32": 1e-5, "fp16": 1e-3}


def _check(cfg, xe, seed):
    from difx_amd.core import FxCore
    offsets = (0, 1, 0)
    data, ctrl = slot(cfg, offsets, seed=seed)
    ref, _ = fo.process_subint(cfg, list(offsets), data, ctrl)
    lay = fo.result_layout(cfg)
    with FxCore(cfg) as core:
        first = core.processdata(offsets, data, ctrl)
        again = core.processdata(offsets, data, ctrl)
    np.testing.assert_array_equal(first.view(np.uint64), again.view(np.uint64))
    e = record_errors(cfg, lay, first.astype(np.complex128), ref)
    print(xe, len(e["cross"]), "records, max", max(e["cross"]), "auto", max(e["auto"]), flush=True)
    assert max(e["cross"]) < BAR[xe] and max(e["auto"]) < BAR[xe]


@pytest.mark.parametrize("xe", ["fp32", "fp16"])
@pytest.mark.parametrize("rows,ffts", [(2, 1), (2, 63), (16, 17), (17, 33), (32, 40), (33, 23), (64, 19)])
def test_row_and_fft_edges(gpu, xe, rows, ffts):
    npol = 2 if rows % 2 == 0 and rows > 2 else 1
    cfg = cf.standard_config(rows // npol, npol, [4800.0], 16.0, 128, subint_ns=ffts * 8000, xengine=xe, seed=31,
                             max_delay_us=50.0)
    _check(cfg, xe, seed=32)


@pytest.mark.parametrize("ffts,chunk", [(700, 0), (700, 264), (9001, 0)])
def test_long_runs_and_chunks(gpu, ffts, chunk):
    """More FFTs than one run of the plain X-engine's sums, in one chunk and in three, and more
    than the weight sums take with their smaller workgroup."""
    cfg = cf.standard_config(4, 2, [4800.0], 16.0, 128, subint_ns=ffts * 8000, xengine="fp32", seed=33,
                             chunk_ffts=chunk, max_delay_us=50.0)
    _check(cfg, "fp32", seed=34)


def test_odd_windows(gpu):
    """13- and 17-channel zoom windows from channels 5 and 110 of 128."""
    cfg = cf.batched_config(3, [(32.0, 128, [4800.0, 4832.0])], [(0, 0, 1.25, 3.25), (0, 1, 27.5, 4.25)],
                            subint_ns=37 * 4000, npol=2, xengine="fp32", seed=35, max_delay_us=50.0)
    _check(cfg, "fp32", seed=36)
