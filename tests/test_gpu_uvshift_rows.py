"""Several phase centres on the 16-bit X-engine where its sums go to the results by either way: read by
the accumulation itself (few products; one and two row tiles, products of rows in both orders, zoom
windows, averaging), or through the reduction (many).  Cross correlations of every phase centre,
autocorrelations and weights against the FP64 oracle, at the parity bars of the FP16 (1e-3) and BF16
(1e-2) visibilities per record."""
import numpy as np
import pytest

import fxoracle as fo
from difx_amd import config as cf
from difx_amd.core import FxCore
from fxcases import case_usb_lsb, record_errors, slot, with_phase_centres
from test_x_targets_cpu import averaged, large_phase_centres

pytestmark = pytest.mark.gpu
OFFS = (0, 1, 0)


def _array(stations, npol, nchan, **kw):
    return lambda xe: with_phase_centres(
        cf.standard_config(stations, npol, [4800.0], 32.0, nchan, subint_ns=24 * nchan * 1000 // 32, xengine=xe, seed=97,
                           max_delay_us=50.0, **kw), P=2, interval_ffts=8, threads=2)


def _swapped(xe):
    """Baselines whose first datastream comes later, and rows in both orders."""
    cfg = _array(5, 2, 128)(xe)
    for b in cfg.baselines[::2]:
        b.ds1, b.ds2 = b.ds2, b.ds1
    return cfg


CASES = {
    "4 stations": _array(4, 2, 256), "33 rows": _array(33, 1, 128), "40 rows": _array(20, 2, 128),
    "averaged": lambda xe: averaged(_array(4, 2, 256)(xe)), "swapped": _swapped,
    "usb x lsb": lambda xe: with_phase_centres(case_usb_lsb(B=24, xengine=xe), P=3),
    "through the reduction": large_phase_centres,
}


@pytest.mark.parametrize("xe,bar", [("fp16", 1e-3), ("bf16", 1e-2)])
@pytest.mark.parametrize("name", sorted(CASES))
def test_either_way(gpu, name, xe, bar):
    cfg = CASES[name](xe)
    data, ctrl = slot(cfg, OFFS, seed=98)
    ref, _ = fo.process_subint(cfg, list(OFFS), data, ctrl)
    lay = fo.result_layout(cfg)
    with FxCore(cfg) as core:
        got = core.processdata(OFFS, data, ctrl)
        again = core.processdata(OFFS, data, ctrl)
    np.testing.assert_array_equal(got.view(np.uint64), again.view(np.uint64))
    e = record_errors(cfg, lay, got.astype(np.complex128), ref)
    print(name, xe, len(e["cross"]), "records, max", max(e["cross"]), "auto", max(e["auto"]), flush=True)
    assert max(e["cross"]) < bar and max(e["auto"]) < bar
