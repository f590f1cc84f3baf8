"""Visibilities with and without the spectral kurtosis on.  FP32 spectra: the same bits.  16-bit
spectra: the F-engine may be another (the per-length kernels instead of the matrix and register
ones), so the spectra round another way here and there; both sets of visibilities are held to the FP16
bar (1e-3 per record) against the FP64 oracle, and turning the kurtosis off again restores the bits."""
import numpy as np
import pytest

import fxoracle as fo
from difx_amd import config as cf
from difx_amd.core import FxCore
from fxcases import record_errors, slot

pytestmark = pytest.mark.gpu
OFFS = (0, 1, 0)


@pytest.mark.parametrize("xe", ["fp32", "fp16"])
@pytest.mark.parametrize("nchan", [1024, 4096])
def test_visibilities_beside_kurtosis(gpu, xe, nchan):
    cfg = cf.standard_config(2, 2, [4800.0], 32.0, nchan, subint_ns=19 * nchan * 1000 // 32, xengine=xe, seed=45,
                             max_delay_us=50.0)
    data, ctrl = slot(cfg, OFFS, seed=46)
    ref, _ = fo.process_subint(cfg, list(OFFS), data, ctrl)
    lay = fo.result_layout(cfg)
    out = []
    with FxCore(cfg) as core:
        for on in (False, True, False):
            core.set_kurtosis(on)
            out.append(core.processdata(OFFS, data, ctrl))
    np.testing.assert_array_equal(out[0].view(np.uint64), out[2].view(np.uint64))
    if xe == "fp32":
        np.testing.assert_array_equal(out[0].view(np.uint64), out[1].view(np.uint64))
    for v in out[:2]:
        e = record_errors(cfg, lay, v.astype(np.complex128), ref)
        assert max(e["cross"]) < (1e-5 if xe == "fp32" else 1e-3) and max(e["auto"]) < (1e-5 if xe == "fp32" else 1e-3)
