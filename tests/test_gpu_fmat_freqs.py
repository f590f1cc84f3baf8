"""The matrix F-engine where a workgroup takes several freqs of its FFTs one after the other (more
FFTs than fill the device): the phasor tables of a freq overlay those of the one before it and the
sample words serve all of them.  8 freqs dual pol with LO and clock offsets, per-pol deltas and phase
offsets and both sidebands, both rotation orders, against the FP64 oracle: spectra of a sample of
FFTs within 2e-5 of their peak and with an rms error no larger than 1.05 times the per-length
kernel's (the two differ in rounding only; 5 % is several times the scatter of either over the
sample's values), visibilities at the FP32 and FP16 bars per record (1e-5, 1e-3)."""
import numpy as np
import pytest

import fxoracle as fo
from difx_amd import config as cf
from difx_amd.core import FxCore
from fxcases import record_errors, slot

pytestmark = pytest.mark.gpu
OFFS = (0, 1, 0)
NFFT = 520                                            # 130 groups of eight FFTs, three freq parts


def _cfg(xe, order, mode):
    cfg = cf.standard_config(2, 2, [4800.0 + 40.0 * k for k in range(8)], 32.0, 1024, subint_ns=NFFT * 32000,
                             xengine=xe, seed=81, max_delay_us=50.0, fringe_rot_order=order, fengine_mode=mode)
    rng = np.random.default_rng(82)
    for f in cfg.freqs[1::3]:
        f.lsb = True
    for d in cfg.datastreams:
        d.lo_offset_hz = [float(rng.choice([0.0, 10.0, -2.5])) for _ in d.recfreqs]
        d.clock_offset_us = [float(rng.uniform(-0.02, 0.02)) for _ in d.recfreqs]
        d.clock_offset_delta_us = [float(rng.uniform(-0.005, 0.005)) for _ in d.recfreqs]
        d.phase_offset_deg = [float(rng.uniform(-90.0, 90.0)) for _ in d.recfreqs]
    return cfg


@pytest.mark.parametrize("order", [0, 1])
def test_several_freqs_per_workgroup(gpu, order):
    cfg = _cfg("fp32", order, 0)
    data, ctrl = slot(cfg, OFFS, seed=83)
    ref, stations = fo.process_subint(cfg, list(OFFS), data, ctrl)
    lay = fo.result_layout(cfg)
    sample = np.r_[0:9, 255:265, NFFT - 9:NFFT]
    rms = []
    for mode in (0, 1):
        e2 = w2 = 0.0
        with FxCore(_cfg("fp32", order, mode)) as core:
            got = core.processdata(OFFS, data, ctrl)
            for d in range(2):
                for b in range(16):
                    for t in sample:
                        w = stations[d].spectra[b][t]
                        e = np.abs(core.getFreqs(d, b, int(t)) - w)
                        assert np.max(e) <= 2e-5 * np.max(np.abs(w)), (mode, d, b, t)
                        e2, w2 = e2 + np.sum(e ** 2), w2 + np.sum(np.abs(w) ** 2)
        rms.append(float(np.sqrt(e2 / w2)))
        e = record_errors(cfg, lay, got.astype(np.complex128), ref)
        assert max(e["cross"]) < 1e-5 and max(e["auto"]) < 1e-5
    print(f"order {order}: spectra rms {rms[0]:.2e}, per-length {rms[1]:.2e}", flush=True)
    assert rms[0] <= 1.05 * rms[1]
    with FxCore(_cfg("fp16", order, 0)) as core:
        e = record_errors(cfg, lay, core.processdata(OFFS, data, ctrl).astype(np.complex128), ref)
    assert max(e["cross"]) < 1e-3 and max(e["auto"]) < 1e-3
