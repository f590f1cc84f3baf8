"""The matrix F-engine against the FP64 oracle where it can go wrong: every FFT length it takes,
fringe rotation orders 0 and 1, both sidebands, band counts that leave a pair of bands short and
that use the upper half of a sample word, per-pol clock deltas and phase offsets (separate
phasor tables in a pair), FFT counts that are not a multiple of its eight FFTs per workgroup,
frames shorter than the stride of its sample loads, and slots with flagged FFTs and invalid
frames.  Spectra: within 2e-5 of the spectrum's peak, the bar of the FP32 F-engine.
Visibilities: the FP32 and FP16 bars per record (1e-5, 1e-3).  The spectra's rms error is also
held to that of the per-length F-engine on the same data."""
import numpy as np
import pytest

import fxoracle as fo
from difx_amd import config as cf
from fxcases import damaged_slot, record_errors, slot

pytestmark = pytest.mark.gpu
OFFS = (0, 1, 0)


def _cfg(nchan, npol=2, nfreq=1, ffts=13, xe="fp32", st=2, **kw):
    return cf.standard_config(st, npol, [4800.0 + 40.0 * k for k in range(nfreq)], 32.0, nchan,
                              subint_ns=ffts * nchan * 1000 // 32, xengine=xe, seed=41, max_delay_us=50.0, **kw)


def _spectra_errors(cfg, data, ctrl, want, ffts):
    """rms and largest error of the spectra of both datastreams, relative to each one's peak and rms."""
    from difx_amd.core import FxCore
    rms, worst = [], 0.0
    with FxCore(cfg) as core:
        got_vis = core.processdata(OFFS, data, ctrl)
        for d in range(2):
            for b in range(len(cfg.datastreams[d].recbands)):
                for t in ffts:
                    w = want[d][b][t]
                    e = core.getFreqs(d, b, t) - w
                    if not np.any(w):
                        assert not np.any(e)
                        continue
                    worst = max(worst, float(np.max(np.abs(e)) / np.max(np.abs(w))))
                    rms.append(float(np.sqrt(np.mean(np.abs(e) ** 2) / np.mean(np.abs(w) ** 2))))
    return got_vis, float(np.mean(rms)), worst


def _check(mk, data_of=slot, ffts=(0, 3, 12)):
    cfg = mk("fp32", 0)
    data, ctrl = data_of(cfg, OFFS, seed=42)
    ref, stations = fo.process_subint(cfg, list(OFFS), data, ctrl)
    want = [s.spectra for s in stations]
    lay = fo.result_layout(cfg)
    vis, rms, worst = _spectra_errors(cfg, data, ctrl, want, ffts)
    _, rms0, _ = _spectra_errors(mk("fp32", 1), data, ctrl, want, ffts)
    e = record_errors(cfg, lay, vis.astype(np.complex128), ref)
    print(f"spectra rms {rms:.2e} (per-length {rms0:.2e}), worst {worst:.2e}; records {max(e['cross']):.2e}", flush=True)
    assert worst < 2e-5 and rms < max(1.5 * rms0, 2.5e-7)
    assert max(e["cross"]) < 1e-5 and max(e["auto"]) < 1e-5
    from difx_amd.core import FxCore
    for xe in ("fp16", "bf16"):
        with FxCore(mk(xe, 0)) as core:
            got = core.processdata(OFFS, data, ctrl)
        e = record_errors(cfg, lay, got.astype(np.complex128), ref)
        bar = {"fp16": 1e-3, "bf16": 1e-2}[xe]
        assert max(e["cross"]) < bar and max(e["auto"]) < bar


NCHAN = [1024]


@pytest.mark.parametrize("nchan", NCHAN)
@pytest.mark.parametrize("order,lsb", [(1, False), (1, True), (0, False), (0, True)])
def test_orders_and_sidebands(gpu, nchan, order, lsb):
    _check(lambda xe, m: _cfg(nchan, xe=xe, fringe_rot_order=order, lsb=lsb, fengine_mode=m))


@pytest.mark.parametrize("nchan", NCHAN)
@pytest.mark.parametrize("npol,nfreq", [(1, 1), (1, 16), (2, 8)])
def test_band_counts(gpu, nchan, npol, nfreq):
    _check(lambda xe, m: _cfg(nchan, npol=npol, nfreq=nfreq, xe=xe, fengine_mode=m))


@pytest.mark.parametrize("nchan", NCHAN)
def test_three_bands_and_pol_tables(gpu, nchan):
    """Two freqs with LO and clock offsets, per-pol deltas and phase offsets; a fractional edge."""
    def mk(xe, m):
        cfg = _cfg(nchan, npol=2, nfreq=2, xe=xe, fengine_mode=m)
        rng = np.random.default_rng(43)
        cfg.freqs[0].freq_mhz = 4800.37
        for d in cfg.datastreams:
            d.lo_offset_hz = [10.0, -2.5]
            d.clock_offset_us = [float(rng.uniform(-0.02, 0.02)) for _ in d.recfreqs]
            d.clock_offset_delta_us = [float(rng.uniform(-0.005, 0.005)) for _ in d.recfreqs]
            d.phase_offset_deg = [float(rng.uniform(-90.0, 90.0)) for _ in d.recfreqs]
        cfg.datastreams[1].recbands = [(lf, "L" if p == "R" else "R") for lf, p in cfg.datastreams[1].recbands]
        return cfg
    _check(mk)


@pytest.mark.parametrize("nchan", NCHAN)
@pytest.mark.parametrize("order", [0, 1])
def test_damaged_slot(gpu, nchan, order):
    _check(lambda xe, m: _cfg(nchan, nfreq=2, xe=xe, fringe_rot_order=order, fengine_mode=m), data_of=damaged_slot,
           ffts=(0, 1, 2, 5, 6, 7, 11, 12))


@pytest.mark.parametrize("nchan", NCHAN)
def test_short_frames(gpu, nchan):
    """16 bands of 1024-byte payloads: 256 samples per frame."""
    _check(lambda xe, m: _cfg(nchan, nfreq=8, xe=xe, payloadbytes=1024, fengine_mode=m))


@pytest.mark.parametrize("nchan", [1024, 4096])
def test_kurtosis_of_16bit_spectra_keeps_the_vector_kernels(gpu, nchan):
    from difx_amd.core import FxCore
    out = []
    for mode in (0, 1):
        cfg = _cfg(nchan, xe="fp16", fengine_mode=mode, fengine_threads=512 if mode and nchan == 4096 else 0)
        data, ctrl = slot(cfg, OFFS, seed=44)
        with FxCore(cfg) as core:
            core.set_kurtosis(True)
            core.processdata(OFFS, data, ctrl)
            out.append(np.stack([core.getKurtosis(d, b, nchan) for d in range(2) for b in range(2)]))
    np.testing.assert_array_equal(out[0], out[1])
