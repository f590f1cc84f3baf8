"""The X-engines' loop over FFTs in several parts, against the FP64 oracle: a subint in ten parts,
in three chunks of which the last is short, in two of which the last has fewer steps than parts
(parts of it stay empty), and two tiles of rows.  The number of parts is read from the tables
first: a case that no longer splits fails.  Bars: the parity bars of the FP32 (1e-5), FP16 (1e-3)
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
    *_, run, parts = extents(cfg)
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
