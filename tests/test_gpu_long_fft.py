"""The per-length F-engine at the lengths with launch forms of their own (8192 points on 1024
threads, complex 4096 points held to 128 registers): every rotation order, both sidebands, two
freqs, an FFT count that fills no unit of eight, on a slot with flagged FFTs and invalid frames
and on a whole one.  Against the FP64 oracle at the FP32 bars: spectra within 2e-5 of their
peak, records within 1e-5."""
import numpy as np
import pytest

import fxoracle as fo
from difx_amd import config as cf
from fxcases import damaged_slot, record_errors, slot

pytestmark = pytest.mark.gpu
OFFS = (0, 1, 0)


@pytest.mark.parametrize("data_of", [slot, damaged_slot])
@pytest.mark.parametrize("nchan,nbits,cplx,order,lsb", [
    (4096, 2, 0, 1, False), (4096, 2, 0, 0, True), (4096, 2, 0, 2, False), (4096, 8, 0, 1, True),
    (8192, 8, 1, 1, False), (8192, 8, 2, 1, False), (4096, 8, 1, 1, True),
    (4096, 8, 2, 1, False), (4096, 8, 1, 2, False)])
def test_long_ffts(gpu, nchan, nbits, cplx, order, lsb, data_of):
    cfg = cf.standard_config(2, 2, [4800.0, 4840.0], 32.0, nchan, subint_ns=13 * nchan * 1000 // 32, nbits=nbits,
                             complex_sampling=cplx, lsb=lsb, fringe_rot_order=order, seed=51, max_delay_us=50.0)
    data, ctrl = data_of(cfg, OFFS, seed=52)
    ref, stations = fo.process_subint(cfg, list(OFFS), data, ctrl)
    from difx_amd.core import FxCore
    with FxCore(cfg) as core:
        got = core.processdata(OFFS, data, ctrl)
        for d in range(2):
            for b in range(4):
                for t in range(13):
                    want = stations[d].spectra[b][t]
                    err = np.max(np.abs(core.getFreqs(d, b, t) - want))
                    assert err <= 2e-5 * np.max(np.abs(want)), (d, b, t)
    e = record_errors(cfg, fo.result_layout(cfg), got.astype(np.complex128), ref)
    assert max(e["cross"]) < 1e-5 and max(e["auto"]) < 1e-5
