"""Jobs whose recorded bands are not all products, on the device against the FP64 oracle: parallel
hands only, a recorded freq that no baseline correlates, and zoom windows without their parents.
A second context of another shape runs before and after on the same device, so that a store
outside one context's buffers would show in the other's results.  Bars: the parity bars of the
FP32 (1e-5) and FP16 (1e-3) visibilities per record."""
import numpy as np
import pytest

import fxoracle as fo
from difx_amd import config as cf
from fxcases import record_errors, slot
from test_x_targets_cpu import averaged, parallel_hands, uncorrelated_freq, zooms_alone

pytestmark = pytest.mark.gpu
OFFS = (0, 1, 0)
BAR = {"fp32": 1e-5, "fp16": 1e-3}


@pytest.mark.parametrize("xe", ["fp32", "fp16"])
@pytest.mark.parametrize("shape", [lambda xe: parallel_hands(xe, nchan=256), lambda xe: uncorrelated_freq(xe, nchan=256),
                                   lambda xe: uncorrelated_freq(xe, npol=2, nchan=256),
                                   lambda xe: averaged(parallel_hands(xe, nchan=256)), zooms_alone],
                         ids=["parallel hands", "uncorrelated freq", "uncorrelated freq dual pol", "averaged", "zooms alone"])
def test_unread_bands(gpu, xe, shape):
    from difx_amd.core import FxCore
    cfg = shape(xe)
    data, ctrl = slot(cfg, OFFS, seed=55)
    ref, _ = fo.process_subint(cfg, list(OFFS), data, ctrl)
    lay = fo.result_layout(cfg)
    other = cf.standard_config(3, 1, [4800.0], 16.0, 128, subint_ns=21 * 8000, xengine="fp32", seed=56, max_delay_us=50.0)
    odata, octrl = slot(other, OFFS, seed=57)
    with FxCore(cfg) as core, FxCore(other) as witness:
        before = witness.processdata(OFFS, odata, octrl)
        got = core.processdata(OFFS, data, ctrl)
        again = core.processdata(OFFS, data, ctrl)
        after = witness.processdata(OFFS, odata, octrl)
    np.testing.assert_array_equal(before.view(np.uint64), after.view(np.uint64))
    np.testing.assert_array_equal(got.view(np.uint64), again.view(np.uint64))
    e = record_errors(cfg, lay, got.astype(np.complex128), ref)
    print(xe, len(e["cross"]), "records, max", max(e["cross"]), "auto", max(e["auto"]), flush=True)
    assert max(e["cross"]) < BAR[xe] and max(e["auto"]) < BAR[xe]
