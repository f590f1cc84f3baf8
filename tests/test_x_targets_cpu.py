"""Where the X-engines store their sums, walked on the host: every store into the product
accumulators and the results, and every read of the accumulators, lies inside its buffer, and
every read finds a stored product.  The tables are those of a host-only context, the same as a
device context's.  The configurations are the ones whose recorded bands are not all products:
parallel hands only, a recorded freq that no baseline correlates, zoom windows with and without
their parents, channel averaging, several phase centres, and rows beyond the matrix tiles."""
import ctypes as C

import pytest

from difx_amd import config as cf
from difx_amd.core import footprint, load_library
from fxcases import case_cfg3, case_offsets, case_usb_lsb, with_phase_centres


def parallel_hands(xe, stations=4, nchan=1024, **kw):
    cfg = cf.standard_config(stations, 2, [4800.0], 32.0, nchan, subint_ns=16 * nchan * 1000 // 32, xengine=xe, seed=51,
                             max_delay_us=50.0, **kw)
    for b in cfg.baselines:
        b.freqs = [(fi, prods[:2]) for fi, prods in b.freqs]
    return cfg


def uncorrelated_freq(xe, npol=1, nchan=1024, **kw):
    """Two recorded freqs, of which the baselines correlate the first."""
    cfg = cf.standard_config(4, npol, [4800.0, 4840.0], 32.0, nchan, subint_ns=16 * nchan * 1000 // 32, xengine=xe,
                             seed=52, max_delay_us=50.0, **kw)
    for b in cfg.baselines:
        b.freqs = b.freqs[:1]
    return cfg


def zooms_alone(xe):
    return cf.batched_config(3, [(32.0, 128, [4800.0, 4832.0])], [(0, 0, 2.0, 4.0), (0, 1, 28.0, 4.0)],
                             subint_ns=16 * 4000, npol=2, xengine=xe, seed=53, max_delay_us=50.0, correlate_parents=False)


def averaged(cfg, n=4):
    for f in cfg.freqs:
        f.chanavg = n
    return cfg


def large_phase_centres(xe):
    """More values than the accumulation reads without the reduction, in two freqs of two row tiles."""
    cfg = cf.standard_config(20, 2, [4800.0, 4840.0], 32.0, 512, subint_ns=24 * 16000, xengine=xe, seed=60,
                             max_delay_us=50.0)
    return with_phase_centres(cfg, P=2, interval_ffts=8, threads=2)


SHAPES = {
    "phase centres, 40 rows": large_phase_centres,
    "parallel hands": parallel_hands,
    "parallel hands, no cross autos": lambda xe: parallel_hands(xe, write_cross_autocorrs=False),
    "parallel hands averaged": lambda xe: averaged(parallel_hands(xe)),
    "uncorrelated freq": uncorrelated_freq,
    "uncorrelated freq dual pol": lambda xe: uncorrelated_freq(xe, npol=2),
    "uncorrelated freq averaged": lambda xe: averaged(uncorrelated_freq(xe)),
    "zooms": lambda xe: case_cfg3(B=16, xengine=xe),
    "zooms alone": zooms_alone,
    "offsets, averaged": lambda xe: case_offsets(B=16, xengine=xe),
    "usb x lsb": lambda xe: case_usb_lsb(B=16, xengine=xe),
    "phase centres": lambda xe: with_phase_centres(parallel_hands(xe)),
    "phase centres, uncorrelated freq": lambda xe: with_phase_centres(uncorrelated_freq(xe, npol=2)),
    "one baseline of two freqs": lambda xe: uncorrelated_freq(xe, nchan=128),
    "72 rows": lambda xe: cf.standard_config(36, 2, [4800.0], 32.0, 128, subint_ns=16 * 4000, xengine=xe, seed=54),
}


def extents(cfg):
    lib = load_library()
    fc, keep = cfg.to_abi()
    h = C.c_void_p()
    assert lib.fxg_create_layout(C.byref(fc), C.byref(h)) == 0, lib.fxg_last_error(None)
    out = (C.c_int64 * 9)()
    lib.fxg_x_extents.argtypes = [C.c_void_p, C.POINTER(C.c_int64)]
    assert lib.fxg_x_extents(h, out) == 0
    lib.fxg_destroy(h)
    return list(out)


@pytest.mark.parametrize("xe", ["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("shape", sorted(SHAPES))
def test_every_target_lies_inside_its_buffer(shape, xe):
    if xe != "fp32" and shape == "72 rows":
        pytest.skip("the 16-bit X-engine takes 64 rows")
    acc, acc_stored, res, res_stored, acc_read, lost, *_ = out = extents(SHAPES[shape](xe))
    print(shape, xe, out)
    assert acc_stored <= acc and acc_read <= acc, (acc_stored, acc_read, acc)
    assert 0 < res_stored <= res
    assert lost == 0


@pytest.mark.parametrize("xe,least", [("fp32", 16), ("fp16", 64), ("bf16", 64)])
@pytest.mark.parametrize("ffts,interval,chunk,longest", [(1200, 0, 0, 1200), (1200, 0, 264, 264), (1200, 40, 0, 40),
                                                        (1200, 100, 0, 100), (1200, 400, 264, 264)])
def test_parts_of_a_run_keep_their_length(xe, least, ffts, interval, chunk, longest):
    """No loop of the X-engine is split into parts shorter than its least, whatever bounds the loop:
    the subint, a chunk of it, or a uv-shift interval with several phase centres."""
    cfg = cf.standard_config(4, 2, [4800.0], 32.0, 128, subint_ns=ffts * 4000, xengine=xe, seed=58, chunk_ffts=chunk)
    if interval:
        with_phase_centres(cfg, P=2, interval_ffts=interval, threads=3)
    *_, run, parts, _ = extents(cfg)
    assert run == longest
    assert 1 <= parts <= max(1, longest // least)


MIB = 1 << 20


@pytest.mark.parametrize("xe", ["fp32", "fp16"])
@pytest.mark.parametrize("stations,npol,nfreq,nchan,avg,centres", [
    (33, 1, 8, 16384, 1, 1), (17, 2, 4, 16384, 1, 1), (33, 1, 8, 16384, 4, 1), (32, 2, 8, 8192, 4, 1), (16, 2, 8, 4096, 1, 3),
    (4, 1, 1, 256, 1, 1), (32, 1, 2, 256, 1, 1), (10, 2, 8, 1024, 1, 1)])
def test_accumulators_are_held_once(xe, stations, npol, nfreq, nchan, avg, centres):
    """The device memory of a context: the chunk's spectra, one set of sums (FP32: a value per
    product; 16-bit: 8 KiB per channel and pair of row tiles) and no more than 200 MiB beside them,
    which holds the parts of a split sum (at most 128 MiB), the products on their way to averaging or
    phase centres (64 MiB, or one freq's) and tables, whatever the job's size."""
    B = 480
    cfg = cf.standard_config(stations, npol, [4800.0 + 70.0 * k for k in range(nfreq)], 32.0, nchan,
                             subint_ns=B * nchan * 1000 // 32, xengine=xe, seed=59, chunk_ffts=64)
    if avg > 1:
        averaged(cfg, avg)
    if centres > 1:
        with_phase_centres(cfg, P=centres, interval_ffts=40, threads=3)
    dev, crl, slot = footprint(cfg)
    n = stations * npol
    tiles = (n + 31) // 32
    spectra = nfreq * nchan * 64 * (8 * n if xe == "fp32" else 4 * 32 * tiles)
    sums = nfreq * nchan * (8 * n * (n + 1) // 2 if xe == "fp32" else 8192 * (tiles * (tiles + 1) // 2))
    fourstep = 1024 * 2 * nchan * 8 if nchan > 4096 else 0      # the four-step F-engine's rows
    print(f"{(dev - spectra - sums) / MIB:.1f} MiB beside spectra and sums; slots {slot / MIB:.1f}, results {8 * crl / MIB:.1f}")
    assert dev <= spectra + sums + 200 * MIB + fourstep


@pytest.mark.parametrize("xe", ["fp32", "fp16"])
def test_parts_hold_the_rows_of_their_group(xe):
    """4 stations dual pol x 256 channels, 8000 FFTs: the parts of the split sums take 64 (FP32) or 128
    values per channel, not whole tiles: no more than 16 MiB beside the spectra, the delay parameters
    and weights."""
    cfg = cf.standard_config(4, 2, [4800.0], 32.0, 256, subint_ns=8000 * 8000, xengine=xe, seed=61)
    *_, parts, _ = extents(cfg)
    assert parts > 8
    dev, _, _ = footprint(cfg)
    spectra = 256 * 8000 * (8 * 8 if xe == "fp32" else 4 * 32)
    print(f"{parts} parts, {(dev - spectra) / MIB:.1f} MiB beside the spectra")
    assert dev <= spectra + 16 * MIB
