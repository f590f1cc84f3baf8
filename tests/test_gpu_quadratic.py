"""Second-order fringe rotation with a quadratic term that matters (a quarter turn of the fringe and
more across an FFT, where the usual delays have next to none) on the register F-engine: against the
FP64 oracle, spectra within 2e-5 of their peak, and their rms error held to 1.05 times that of the
per-length kernel on the same data.  Real 2-bit and complex 8-bit samples, every FFT length."""
import numpy as np
import pytest

import fxoracle as fo
from difx_amd import config as cf
from fxcases import slot

pytestmark = pytest.mark.gpu
OFFS = (0, 1, 0)
FFTS = 9


def _cfg(nchan, cplx, turns, mode):
    cfg = cf.standard_config(2, 1, [4800.0], 32.0, nchan, subint_ns=FFTS * nchan * 1000 // 32, xengine="fp32", seed=95,
                             fringe_rot_order=2, fengine_mode=mode, nbits=8 if cplx else 2, complex_sampling=cplx)
    span = nchan / 32e6                                # seconds of one FFT
    for k, d in enumerate(cfg.datastreams):            # c (t - 1 s)^2: no large delay near the subint
        c = (1 - 2 * k) * turns / (4800.0 * span ** 2)
        d.model[:, :] = 0.0
        d.model[:, :3] = [c + 3.1 * k, -2 * c + 0.4, c]
    return cfg


@pytest.mark.parametrize("turns", [0.25, 0.7])
@pytest.mark.parametrize("nchan,cplx", [(2048, 0), (4096, 0), (8192, 0), (16384, 0), (4096, 1), (16384, 1)])
def test_quadratic_term(gpu, nchan, cplx, turns):
    from difx_amd.core import FxCore
    cfg = _cfg(nchan, cplx, turns, 0)
    data, ctrl = slot(cfg, OFFS, seed=96)
    _, stations = fo.process_subint(cfg, list(OFFS), data, ctrl)
    rms = []
    for mode in (0, 1):
        e2 = w2 = 0.0
        with FxCore(_cfg(nchan, cplx, turns, mode)) as core:
            core.processdata(OFFS, data, ctrl)
            for d in range(2):
                for t in range(FFTS):
                    w = stations[d].spectra[0][t]
                    e = np.abs(core.getFreqs(d, 0, t) - w)
                    assert np.max(e) <= 2e-5 * np.max(np.abs(w)), (mode, d, t)
                    e2, w2 = e2 + np.sum(e ** 2), w2 + np.sum(np.abs(w) ** 2)
        rms.append(float(np.sqrt(e2 / w2)))
    print(f"spectra rms {rms[0]:.2e}, per-length {rms[1]:.2e}", flush=True)
    assert rms[0] <= 1.05 * rms[1]
