"""Rounding of the plain FP32 X-engine's short sums: its visibilities are no further from 64-bit
sums of the spectra that it read than a plain FP32 sum of four consecutive parts of them is, the
order of the lane-per-channel sums (both measured here over the same spectra, the FP32 sum in numpy).
24 to 250 FFTs, one baseline to ten stations.  The bar is 1.0 plus 5 % for the scatter of a mean over
some thousand values."""
import numpy as np
import pytest

from difx_amd import config as cf
from difx_amd.core import FxCore
from fxcases import slot
import fxoracle as fo

pytestmark = pytest.mark.gpu
OFFS = (0, 1, 0)


def _fp32_parts(x, y):
    """sum of x conj(y) over FFTs in FP32: four consecutive parts, each in order, then added."""
    n = len(x)
    re = im = None
    for q in range(4):
        r = i = np.zeros(x.shape[1], np.float32)
        for t in range(n * q // 4, n * (q + 1) // 4):
            r = (r + x[t].real * y[t].real) + x[t].imag * y[t].imag
            i = (i + x[t].imag * y[t].real) - x[t].real * y[t].imag
        re, im = (r, i) if re is None else (re + r, im + i)
    return re.astype(np.float64) + 1j * im


@pytest.mark.parametrize("stations,npol,ffts", [(2, 1, 24), (3, 1, 30), (2, 1, 63), (2, 1, 120), (5, 2, 63), (2, 1, 250), (12, 2, 24), (40, 1, 24)])
def test_short_sums(gpu, stations, npol, ffts):
    cfg = cf.standard_config(stations, npol, [4800.0], 16.0, 512, subint_ns=ffts * 32000, xengine="fp32", seed=91,
                             max_delay_us=50.0)
    lay = fo.result_layout(cfg)
    e2 = p2 = 0.0
    for seed in (92, 93, 94):
        data, ctrl = slot(cfg, OFFS, seed=seed)
        with FxCore(cfg) as core:
            got = core.processdata(OFFS, data, ctrl)
            spec = [[np.stack([core.getFreqs(d, b, t) for t in range(ffts)]) for b in range(npol)] for d in range(stations)]
        for j, bl in enumerate(cfg.baselines):
            for fi, prods in bl.freqs:
                off = lay.baseline_off[fi, j]
                for p, (b1, b2) in enumerate(prods):
                    x, y = spec[bl.ds1][b1], spec[bl.ds2][b2]
                    want = np.sum(x.astype(np.complex128) * np.conj(y.astype(np.complex128)), axis=0)
                    e2 += float(np.sum(np.abs(got[off + p * 512: off + (p + 1) * 512] - want) ** 2))
                    p2 += float(np.sum(np.abs(_fp32_parts(x, y) - want) ** 2))
    print(f"{stations} stations, {ffts} FFTs: error {np.sqrt(e2 / p2):.3f} of the plain FP32 sum's", flush=True)
    assert e2 <= 1.05 ** 2 * p2
