"""The register F-engine (4096- to 32768-point FFTs of real 2-bit and complex 8-bit samples) against the FP64
oracle where it can go wrong: every rotation order and both sidebands, one band per freq and
sixteen bands, per-pol clock deltas and phase offsets (separate phasor tables), frames shorter
than the stride of its sample loads, an FFT count that fills no workgroup, and slots with flagged
FFTs and invalid frames.  Spectra: within 2e-5 of the spectrum's peak, the bar of the FP32
F-engine, and their rms error held to that of the per-length kernel on the same data.
Visibilities: the FP32 and FP16 bars per record (1e-5, 1e-3)."""
import numpy as np
import pytest

import fxoracle as fo
from difx_amd import config as cf
from fxcases import damaged_slot, record_errors, slot

pytestmark = pytest.mark.gpu
OFFS = (0, 1, 0)
NCHAN = [2048, 4096, 8192, 16384]


def _cfg(nchan, npol=2, nfreq=1, ffts=5, xe="fp32", **kw):
    return cf.standard_config(2, npol, [4800.0 + 40.0 * k for k in range(nfreq)], 32.0, nchan,
                              subint_ns=ffts * nchan * 1000 // 32, xengine=xe, seed=61, max_delay_us=50.0, **kw)


def _check(mk, data_of=slot):
    from difx_amd.core import FxCore
    cfg = mk("fp32", 0)
    data, ctrl = data_of(cfg, OFFS, seed=62)
    ref, stations = fo.process_subint(cfg, list(OFFS), data, ctrl)
    lay = fo.result_layout(cfg)
    rms = []
    for mode in (0, 1):
        e2 = w2 = 0.0
        with FxCore(mk("fp32", mode)) as core:
            got = core.processdata(OFFS, data, ctrl)
            for d in range(2):
                for b in range(len(cfg.datastreams[d].recbands)):
                    for t in range(5):
                        w = stations[d].spectra[b][t]
                        e = np.abs(core.getFreqs(d, b, t) - w)
                        assert np.max(e) <= 2e-5 * np.max(np.abs(w)), (mode, d, b, t)
                        e2, w2 = e2 + np.sum(e ** 2), w2 + np.sum(np.abs(w) ** 2)
        rms.append(float(np.sqrt(e2 / w2)))
        e = record_errors(cfg, lay, got.astype(np.complex128), ref)
        assert max(e["cross"]) < 1e-5 and max(e["auto"]) < 1e-5
    print(f"spectra rms {rms[0]:.2e}, per-length {rms[1]:.2e}", flush=True)
    assert rms[0] <= 1.05 * rms[1]
    with FxCore(mk("fp16", 0)) as core:
        e = record_errors(cfg, lay, core.processdata(OFFS, data, ctrl).astype(np.complex128), ref)
    assert max(e["cross"]) < 1e-3 and max(e["auto"]) < 1e-3


@pytest.mark.parametrize("nchan", NCHAN)
@pytest.mark.parametrize("order,lsb", [(1, False), (1, True), (0, False), (0, True), (2, False)])
def test_orders_and_sidebands(gpu, nchan, order, lsb):
    _check(lambda xe, m: _cfg(nchan, xe=xe, fringe_rot_order=order, lsb=lsb, fengine_mode=m))


@pytest.mark.parametrize("nchan", NCHAN)
@pytest.mark.parametrize("npol,nfreq", [(1, 1), (2, 8)])
def test_band_counts(gpu, nchan, npol, nfreq):
    _check(lambda xe, m: _cfg(nchan, npol=npol, nfreq=nfreq, xe=xe, fengine_mode=m))


@pytest.mark.parametrize("nchan", NCHAN)
def test_pol_tables(gpu, nchan):
    """Two freqs with LO and clock offsets, per-pol deltas and phase offsets; a fractional edge."""
    def mk(xe, m):
        cfg = _cfg(nchan, nfreq=2, xe=xe, fengine_mode=m)
        rng = np.random.default_rng(63)
        cfg.freqs[0].freq_mhz = 4800.37
        for d in cfg.datastreams:
            d.lo_offset_hz = [10.0, -2.5]
            d.clock_offset_us = [float(rng.uniform(-0.02, 0.02)) for _ in d.recfreqs]
            d.clock_offset_delta_us = [float(rng.uniform(-0.005, 0.005)) for _ in d.recfreqs]
            d.phase_offset_deg = [float(rng.uniform(-90.0, 90.0)) for _ in d.recfreqs]
        return cfg
    _check(mk)


@pytest.mark.parametrize("nchan", NCHAN)
@pytest.mark.parametrize("order,payload", [(0, 8000), (1, 8000), (2, 8000), (1, 1024)])
def test_damaged_slot(gpu, nchan, order, payload):
    """Payloads of 1024 bytes with 16 bands: 256 samples per frame."""
    _check(lambda xe, m: _cfg(nchan, nfreq=8 if payload < 8000 else 2, xe=xe, fringe_rot_order=order,
                              payloadbytes=payload, fengine_mode=m), data_of=damaged_slot)


@pytest.mark.parametrize("nchan", NCHAN)
def test_short_frames(gpu, nchan):
    _check(lambda xe, m: _cfg(nchan, nfreq=8, xe=xe, payloadbytes=1024, fengine_mode=m))


@pytest.mark.parametrize("nchan", [4096, 8192, 16384, 32768])
@pytest.mark.parametrize("cplx,lsb,order,data_of", [(1, False, 1, slot), (1, True, 1, damaged_slot), (2, False, 1, damaged_slot),
                                                    (1, True, 2, damaged_slot)])
def test_complex(gpu, nchan, cplx, lsb, order, data_of):
    _check(lambda xe, m: _cfg(nchan, xe=xe, nbits=8, complex_sampling=cplx, lsb=lsb, fringe_rot_order=order,
                              fengine_mode=m), data_of=data_of)
