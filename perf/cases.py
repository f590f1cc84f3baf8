"""Workloads of the FX correlator library whose times are compared between versions.

Every case is one call path a program takes through the public entry points: a subint through
`FxCore.processdata_device` (slot buffers and results resident on the device), through
`FxCore.processdata` (host buffers in and out, the drop-in for Core::processdata), a subint with
its side products (spectral kurtosis and phase-cal tones), and the corner turn of one segment
of VDIF threads.  `listed()` holds the repository's own configurations at their real lengths,
`draw()` more cases of the same ranges, `work()` the bytes and operations a pass cannot do
without, and `exact()` the same results in 64 bits from plain torch.
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

from difx_amd import config as cf
from difx_amd import synth
from difx_amd.core import FxCore
from difx_amd.vdifmux import VDIFMuxer

OFFSETS = (0, 1, 0)                 # {scan, sec, ns} of every case's subint
HIMAG = 3.3359                      # outer level of a 2-bit sample
_shared = {}


def _stream() -> int:
    """The one stream a program runs its subints on, as a hipStream_t."""
    if "stream" not in _shared:
        _shared["stream"] = torch.cuda.Stream()
    return _shared["stream"].cuda_stream


# ---- the cases -----------------------------------------------------------------------------

def _fx(name="", stations=4, pols=2, freqs=1, bw=32, nchan=1024, ffts=1000, nbits=2, cplx=0, fmt="VDIF",
        xengine="fp16", order=1, lsb=False, bad=0, host=False, side=False):
    """A standard array: `stations` datastreams of pols x freqs bands of bw MHz; `bad` frames
    in a thousand are flagged invalid by the recorder; `host`: host buffers in and out; `side`:
    spectral kurtosis and a 1 MHz phase-cal comb as well."""
    c = dict(kind="fx", stations=stations, pols=pols, freqs=freqs, bw=bw, nchan=nchan, ffts=ffts, nbits=nbits,
             cplx=cplx, fmt=fmt, xengine=xengine, order=order, lsb=lsb, bad=bad, host=host, side=side)
    if name:
        c["name"] = name
    return c


def _uneven(name="", stations=16, bands="long", ffts=2000, xengine="fp16", bad=0):
    """Uneven bands with zoom windows: one datastream per station and bandwidth."""
    c = dict(kind="uneven", stations=stations, bands=bands, ffts=ffts, xengine=xengine, bad=bad)
    if name:
        c["name"] = name
    return c


def _mux(name="", threads=16, nbits=2, slots=1000, payload=8000, lost=0):
    """One station segment of single-channel VDIF threads; `lost` frames in a thousand never
    arrived."""
    c = dict(kind="mux", threads=threads, nbits=nbits, slots=slots, payload=payload, lost=lost)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # a fringe check on one baseline: the smallest call, 0.5 ms of one 16 MHz band
        _fx("fringe_check_2st", stations=2, pols=1, freqs=1, bw=16, nchan=128, ffts=63, xengine="fp32"),
        # the drop-in call with host buffers: 0.1 s of the 4-station single-band configuration
        _fx("host_4st", stations=4, pols=1, freqs=1, nchan=256, ffts=12500, xengine="fp32", host=True),
        # the 4-station single-band configuration at its 1 s subint, plain FP32 X-engine
        _fx("plain_4st_1s", stations=4, pols=1, freqs=1, nchan=256, ffts=125000, xengine="fp32"),
        # the 10-station array, 8 x 32 MHz dual pol, 0.5 s, plain FP32; a few frames flagged invalid
        _fx("plain_10st", stations=10, freqs=8, ffts=15625, xengine="fp32", bad=1),
        # the benchmark's workload: 16 stations, 8 x 32 MHz dual pol, 0.5 s, FP16 matrix X-engine
        _fx("array_16st_fp16", stations=16, freqs=8, ffts=15625, xengine="fp16"),
        # 64 stations of complex 8-bit samples, 4096-point FFTs, 1 s, BF16 matrix X-engine
        _fx("complex8_64st_bf16", stations=64, pols=1, bw=16, nchan=4096, ffts=3906, nbits=8, cplx=1,
            xengine="bf16"),
        # uneven bands: 4 x 64, 4 x 32 and 8 x 8 MHz with six zooms (4096- to 32768-point FFTs)
        _uneven("uneven_16st", stations=16, bands="long", ffts=1001),
        # jobs of the serving stream: many stations with short FFTs, few with long ones
        _fx("serve_32st_256ch", stations=32, freqs=2, nchan=256, ffts=8001, xengine="fp16"),
        _fx("serve_8st_4096ch", stations=8, freqs=4, nchan=4096, ffts=1000, xengine="fp16"),
        # post-F fringe rotation on Mark5B recordings, an odd number of FFTs
        _fx("postf_8st_mark5b", stations=8, freqs=4, nchan=512, ffts=6251, fmt="MARK5B", xengine="fp16", order=0),
        # a pulsar-band monitor: kurtosis of every band and phase-cal tones beside the subint
        _fx("side_4st", stations=4, freqs=2, nchan=512, ffts=6250, xengine="fp32", side=True),
        # half a second of one station's 16-thread recording turned into 16-channel frames
        _mux("corner_turn_16", threads=16, slots=1000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _cost(c):
    """Rough cost of a case: input samples, plus the products' share."""
    if c["kind"] == "mux":
        return c["threads"] * c["slots"] * c["payload"] * 2
    w = work(c)
    return w["flops"]


def draw(rng):
    kind = rng.choice(["fx"] * 7 + ["uneven", "side", "mux"])
    if kind == "mux":
        threads = rng.choice([2, 4, 8, 16])
        return _mux(threads=threads, nbits=2 if threads > 8 else rng.choice([2, 4] if threads > 2 else [2, 8]),
                    slots=_log_int(rng, 9, 2000), payload=rng.choice([1000, 5000, 8000]), lost=rng.choice([0, 0, 2]))
    if kind == "uneven":
        bands = rng.choice(["long", "short"])
        c = _uneven(stations=rng.randint(2, 12), bands=bands,
                    ffts=_log_int(rng, 40, 500) if bands == "long" else _log_int(rng, 100, 8000),
                    xengine=rng.choice(["fp32", "fp16"]), bad=rng.choice([0, 0, 1]))
    elif kind == "side":
        c = _fx(stations=rng.randint(2, 8), pols=2, freqs=rng.choice([1, 2]), nchan=rng.choice([256, 512, 1024]),
                ffts=_log_int(rng, 500, 8000), xengine=rng.choice(["fp32", "fp16"]), side=True)
    elif rng.random() < 0.15:                        # complex 8-bit sampling
        c = _fx(stations=_log_int(rng, 2, 64), pols=1, freqs=rng.choice([1, 2]), bw=rng.choice([16, 32]),
                nchan=rng.choice([256, 1024, 4096, 8192]), ffts=_log_int(rng, 64, 8000), nbits=8, cplx=1,
                xengine=rng.choice(["fp32", "fp16", "bf16"]))
    elif rng.random() < 0.15:                        # real 8-bit sampling
        c = _fx(stations=_log_int(rng, 2, 16), pols=rng.choice([1, 2]), freqs=rng.choice([1, 2]), bw=16,
                nchan=rng.choice([256, 512, 2048]), ffts=_log_int(rng, 64, 8000), nbits=8,
                xengine=rng.choice(["fp32", "fp16"]), order=rng.choice([0, 1]))
    else:
        pols = rng.choice([1, 2, 2])
        c = _fx(stations=_log_int(rng, 2, 32), pols=pols, freqs=rng.choice([1, 2, 4, 8]), bw=rng.choice([8, 16, 32, 64]),
                nchan=rng.choice([128, 256, 512, 1024, 1024, 2048, 4096, 8192, 16384]), ffts=_log_int(rng, 24, 60000),
                fmt=rng.choice(["VDIF", "VDIF", "MARK5B"]), xengine=rng.choice(["fp32", "fp16", "fp16", "bf16"]),
                order=rng.choice([0, 1, 1, 1, 2]), lsb=rng.random() < 0.25, bad=rng.choice([0, 0, 0, 1]),
                host=rng.random() < 0.1)
    if c.get("fmt") == "MARK5B" and c["pols"] * c["freqs"] * c["bw"] > 256:
        c["fmt"] = "VDIF"                            # a Mark5B frame has to last whole nanoseconds
    top = 0.6 * _cost(next(x for x in listed() if x["name"] == "array_16st_fp16"))
    if c.get("host"):
        top /= 40                                    # host buffers: at most about 100 MB
    while _cost(c) > top and c["ffts"] > 24:
        c["ffts"] = max(24, int(c["ffts"] * 0.71))
    while _cost(c) > top:
        c["stations"] = max(2, c["stations"] // 2)
    return c


# ---- configurations and inputs -------------------------------------------------------------

def _config(c):
    if c["kind"] == "uneven":
        if c["bands"] == "long":
            groups = [(64.0, 16384, [4800.0 + 64.0 * k for k in range(4)]),
                      (32.0, 8192, [5200.0 + 32.0 * k for k in range(4)]),
                      (8.0, 2048, [5400.0 + 8.0 * k for k in range(8)])]
            zooms = [(0, 0, 10.0, 2.0), (0, 2, 30.0, 0.5), (1, 1, 4.0, 1.0), (1, 3, 20.0, 2.0),
                     (2, 0, 1.0, 0.5), (2, 5, 3.0, 2.0)]
        else:
            groups = [(32.0, 512, [4800.0, 4832.0]), (8.0, 128, [4900.0, 4908.0]), (64.0, 1024, [5000.0])]
            zooms = [(0, 1, 4.0, 2.0), (0, 0, 10.0, 1.0), (1, 1, 2.0, 0.5), (2, 0, 20.0, 2.0)]
        fft_ns = int(1000 * groups[0][1] // groups[0][0])
        return cf.batched_config(c["stations"], groups, zooms, subint_ns=c["ffts"] * fft_ns, xengine=c["xengine"],
                                 seed=20261203, max_delay_us=300.0)
    fft_ns = 1000 * c["nchan"] // c["bw"]
    cfg = cf.standard_config(c["stations"], c["pols"], [4800.0 + 2 * c["bw"] * k for k in range(c["freqs"])],
                             float(c["bw"]), c["nchan"], subint_ns=c["ffts"] * fft_ns, nbits=c["nbits"],
                             complex_sampling=c["cplx"], seed=20261205, xengine=c["xengine"], lsb=c["lsb"],
                             fringe_rot_order=c["order"], max_delay_us=300.0)
    for ds in cfg.datastreams:
        if c["fmt"] == "MARK5B":
            ds.format, ds.headerbytes, ds.payloadbytes = "MARK5B", 16, 10000
        if c["side"]:
            ds.phasecal_interval_hz = 1_000_000
    return cfg


def _byte_table(fmt, device):
    """Inverse distribution of a byte of four 2-bit samples, over 16-bit random numbers: the
    levels of Gaussian noise with thresholds at 0.95 sigma."""
    p_hi = 0.5 * math.erfc(0.95 / math.sqrt(2.0))
    prob = np.array([p_hi, 0.5 - p_hi, 0.5 - p_hi, p_hi])            # by level, low to high
    code = [0, 2, 1, 3] if fmt == "MARK5B" else [0, 1, 2, 3]
    pc = np.zeros(4)
    for level, q in enumerate(code):
        pc[q] = prob[level]
    b = np.arange(256)
    pb = pc[b & 3] * pc[(b >> 2) & 3] * pc[(b >> 4) & 3] * pc[b >> 6]
    edges = np.floor(np.cumsum(pb) * 65536 + 0.5).astype(np.int64)
    return torch.from_numpy(np.searchsorted(edges, np.arange(65536), side="right").clip(0, 255).astype(np.uint8)).to(device)


def _headers(ds, nframes, first, invalid):
    w = np.zeros((nframes, ds.headerbytes // 4), dtype=np.uint32)
    f = first + np.arange(nframes)
    if ds.format == "MARK5B":
        w[:, 0] = 0xABADDEED
        w[:, 1] = (f & 0x7FFF) | (invalid.astype(np.uint32) << 15)
    else:
        w[:] = synth.vdif_header(0, 0, ds.framebytes, len(ds.recbands), ds.nbits, bool(ds.complex_sampling)).view(np.uint32)
        w[:, 0] = invalid.astype(np.uint32) << 31
        w[:, 1] = f & 0xFFFFFF
    return torch.from_numpy(w.view(np.uint8).reshape(nframes, ds.headerbytes))


def _slot(cfg, bad, seed, dev):
    """Device slot buffers, their lengths, the control words and each buffer's invalid frames."""
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    rng = np.random.default_rng(seed)
    bufs, nbytes, ctrl, flags = [], [], [], []
    table = {}
    for d, ds in enumerate(cfg.datastreams):
        start_ns = synth.buffer_start_ns(cfg, d, OFFSETS)
        nframes = synth.slot_bytes(cfg, d, OFFSETS, start_ns) // ds.framebytes
        pay = ds.framebytes - ds.headerbytes
        frame_ns = int(round(synth.samples_per_frame(ds) * cfg.sampletime_us(d) * 1000.0))
        invalid = rng.random(nframes) < bad / 1000.0
        buf = torch.empty((nframes, ds.framebytes), dtype=torch.uint8, device=dev)
        if ds.nbits == 2:
            if ds.format not in table:
                table[ds.format] = _byte_table(ds.format, dev)
            r = torch.randint(0, 65536, (nframes * pay,), dtype=torch.int32, device=dev, generator=g)
            buf[:, ds.headerbytes:] = table[ds.format].index_select(0, r).view(nframes, pay)
        else:
            x = torch.randn((nframes, pay), device=dev, generator=g)
            buf[:, ds.headerbytes:] = x.mul_(20.0).add_(128.0).round_().clamp_(0, 255).to(torch.uint8)
        buf[:, : ds.headerbytes] = _headers(ds, nframes, start_ns // frame_ns, invalid).to(dev)
        bufs.append(buf.view(-1))
        nbytes.append(nframes * ds.framebytes)
        ctrl.append(synth.control_words(cfg, d, OFFSETS, start_ns))
        flags.append(invalid)
    return bufs, nbytes, ctrl, flags


def _mux_input(c, seed, dev):
    """The segment's frames in arrival order, and the reference time."""
    n, ns, fps = c["threads"], c["slots"], 2000
    tfb = c["payload"] + 32
    rng = np.random.default_rng(seed)
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    s, t = np.repeat(np.arange(ns), n), np.tile(np.arange(n), ns)
    hdr = np.zeros((ns * n, 8), dtype=np.uint32)
    hdr[:, 0] = 5000 + s // fps
    hdr[:, 1] = (s % fps) | (40 << 24)
    hdr[:, 2] = tfb // 8
    hdr[:, 3] = 0x4142 | (t << 16) | ((c["nbits"] - 1) << 26)
    # threads arrive interleaved, a frame time or two out of order
    order = np.argsort(s + rng.uniform(0, 2, ns * n), kind="stable")
    keep = order[(rng.random(ns * n) >= c["lost"] / 1000.0) | (order < n)]
    fr = torch.randint(0, 256, (len(keep), tfb), dtype=torch.uint8, device=dev, generator=g)
    fr[:, :32] = torch.from_numpy(hdr[keep].view(np.uint8).reshape(-1, 32)).to(dev)
    return fr.view(-1), 58849 * 86400 + 5000, fps, tfb


class _State:
    def __del__(self):
        core = getattr(self, "core", None)
        if core is not None:
            torch.cuda.synchronize()
            core.close()


def prepare(case, seed):
    dev = torch.device("cuda:0")
    s = _State()
    s.case = case
    if case["kind"] == "mux":
        s.frames, ref, fps, tfb = _mux_input(case, seed, dev)
        s.mux = VDIFMuxer(case["threads"], tfb, fps, case["nbits"], list(range(case["threads"])))
        s.mux.set_reference(ref, 0)
        s.out = torch.zeros(case["slots"] * s.mux.outputframebytes, dtype=torch.uint8, device=dev)
        return s
    cfg = _config(case)
    s.bufs, s.nbytes, s.ctrl, _ = _slot(cfg, case["bad"], seed, dev)
    s.core = FxCore(cfg)
    if case.get("host"):
        s.bufs = [b.cpu().numpy() for b in s.bufs]
        return s
    s.ptrs = [b.data_ptr() for b in s.bufs]
    s.res = torch.zeros(s.core.coreresultlength, dtype=torch.complex64, device=dev)
    if case.get("side"):
        s.core.set_kurtosis(True)
    s.stream = _stream()
    torch.cuda.synchronize()                         # the inputs are made on another stream
    return s


def run(state):
    c = state.case
    if c["kind"] == "mux":
        out, nbytes = state.mux.multiplex(state.frames, c["slots"], out=state.out, start=0)
        return {"frames": out, "bytes": nbytes}
    if c.get("host"):
        return state.core.processdata(OFFSETS, state.bufs, state.ctrl)
    state.core.processdata_device(OFFSETS, state.ptrs, state.nbytes, state.ctrl, state.res.data_ptr(), state.stream)
    if c.get("side"):
        sk = [state.core.getKurtosis(d, b, c["nchan"]) for d, ds in enumerate(state.core.cfg.datastreams)
              for b in range(len(ds.recbands))]
        return {"results": state.res, "kurtosis": np.stack(sk)}
    return state.res


# ---- what a pass cannot do without ---------------------------------------------------------

def work(case):
    if case["kind"] == "mux":
        frame = case["payload"] + 32
        kept = case["threads"] * case["slots"] * (1 - case["lost"] / 1000.0)
        return {"bytes": kept * frame + case["slots"] * (case["payload"] * case["threads"] + 32), "flops": 0}
    cfg = _config(case)
    B = cfg.blockspersend()
    nbytes = flops = results = 0.0
    for d, ds in enumerate(cfg.datastreams):
        L, C, nb = cfg.fftchannels(d), cfg.freqs[ds.recfreqs[0]].nchan, len(ds.recbands)
        nbytes += B * L * nb * ds.nbits * (2 if ds.complex_sampling else 1) / 8
        half = 0.5 if cfg.fringe_rot_order == 0 and not ds.complex_sampling else 1.0
        fft = half * 5 * L * math.log2(L) + (0 if cfg.fringe_rot_order == 0 else 2 * L) + 6 * C
        flops += B * nb * (fft + 8 * C * (2 if len({p for _, p in ds.recbands}) > 1 else 1))
        results += nb * C * (2 if len({p for _, p in ds.recbands}) > 1 else 1)
    for b in cfg.baselines:
        for fi, prods in b.freqs:
            flops += 8.0 * B * cfg.freqs[fi].nchan * len(prods)
            results += cfg.freqs[fi].nchan * len(prods)
    return {"bytes": nbytes + 8 * results, "flops": flops}


# ---- the same results in 64 bits -----------------------------------------------------------

def _delays(cfg, d, B):
    """Per FFT of datastream d, in double: first sample, fractional error (us, rounded to float
    as the correlator does), and the delay polynomial across the FFT."""
    ds = cfg.datastreams[d]
    C, L = cfg.freqs[ds.recfreqs[0]].nchan, cfg.fftchannels(d)
    dt = cfg.sampletime_us(d)
    t0 = OFFSETS[1] + OFFSETS[2] / 1e9
    span = B * C / cfg.freqs[ds.recfreqs[0]].bw_mhz / 1e6
    m0, m1, m2 = (sum(ds.model[0, k] * t ** k for k in range(ds.model_order + 1)) for t in (t0, t0 + span / 2, t0 + span))
    q0, q1, q2 = (2 * m0 - 4 * m1 + 2 * m2) / B ** 2, (-3 * m0 + 4 * m1 - m2) / B, m0
    i = np.arange(B, dtype=np.float64)
    at = lambda x: q0 * x * x + q1 * x + q2                           # noqa: E731
    start = synth.buffer_start_ns(cfg, d, OFFSETS)
    sec, ns = start // 10 ** 9, start % 10 ** 9
    t = (OFFSETS[1] - sec) * 1e6 + (OFFSETS[2] - ns) / 1000.0 + i * L * dt - at(i + 0.5)
    n0 = np.trunc(t / dt + 0.5).astype(np.int64)
    fse = (t - n0 * dt).astype(np.float32).astype(np.float64)
    if cfg.fringe_rot_order == 1:
        a = at(i + 1) - at(i)
        poly = (np.zeros(B), a, at(i) + (at(i + 0.5) - (a / 2 + at(i))) / 3)
    elif cfg.fringe_rot_order == 2:
        poly = (np.full(B, q0), q1 + 2 * i * q0, q2 + i * q1 + i * i * q0)
    else:
        poly = (np.zeros(B), np.zeros(B), at(i + 0.5))
    return n0, fse, poly, int(round((sec * 1e9 + ns) / (dt * 1000)))


def _turn(ph):
    """exp(2 pi i ph) of a phase in turns."""
    a = 2 * math.pi * (ph - torch.floor(ph))
    return torch.complex(torch.cos(a), torch.sin(a))


def _exact_subint(case, seed):
    dev = torch.device("cuda:0" if torch.cuda.is_available() else "cpu")
    cfg = _config(case)
    B, order = cfg.blockspersend(), cfg.fringe_rot_order
    bufs, _, _, flags = _slot(cfg, case["bad"], seed, dev)
    nds = len(cfg.datastreams)
    delays = [_delays(cfg, d, B) for d in range(nds)]
    side = bool(case.get("side"))
    lut = {"VDIF": [-HIMAG, -1.0, 1.0, HIMAG], "MARK5B": [-HIMAG, 1.0, -1.0, HIMAG]}
    # FP32 levels are what the sample format defines
    lut = {k: torch.tensor(v, dtype=torch.float32, device=dev).double() for k, v in lut.items()}
    lut8 = ((torch.arange(256, dtype=torch.float64) - 128.0) / 3.3).float().double().to(dev)
    weights = [np.zeros(B) for _ in range(nds)]
    # datastreams that share their freqs are correlated together
    sets = {}
    for d, ds in enumerate(cfg.datastreams):
        sets.setdefault(tuple(ds.recfreqs), []).append(d)
    V, rows, kurt, tones = {}, {}, {}, {}
    for fl, dd in sets.items():
        d0 = cfg.datastreams[dd[0]]
        L, C = cfg.fftchannels(dd[0]), cfg.freqs[fl[0]].nchan
        nb, spf = len(d0.recbands), synth.samples_per_frame(d0)
        pay = d0.framebytes - d0.headerbytes
        per = {lf: [b for b, (x, _) in enumerate(d0.recbands) if x == lf] for lf in range(len(fl))}
        T = max(1, min(B, int((3 << 30) // (16 * L * len(dd) * max(len(v) for v in per.values())))))
        loads = [bufs[d].view(-1, d0.framebytes)[:, d0.headerbytes:].contiguous().view(-1) for d in dd]
        good = [torch.from_numpy(~flags[d]).to(dev) for d in dd]
        ns = torch.arange(L, device=dev)
        cs = torch.arange(C, device=dev, dtype=torch.float64)
        for lf, fi in enumerate(fl):
            nr = len(dd) * len(per[lf])
            V[fl, lf] = torch.zeros((C, nr, nr), dtype=torch.complex128, device=dev)
            for k, d in enumerate(dd):
                for m, b in enumerate(per[lf]):
                    rows[d, b] = (fl, lf, k * len(per[lf]) + m)
                    kurt[d, b] = torch.zeros((2, C), dtype=torch.float64, device=dev)
                    tones[d, b] = torch.zeros(2 * int(d0.phasecal_interval_hz and cfg.freqs[fi].bw_mhz), dtype=torch.float64, device=dev)
        for t0 in range(0, B, T):
            t1 = min(B, t0 + T)
            for lf, fi in enumerate(fl):
                fr = cfg.freqs[fi]
                X = torch.empty((len(dd) * len(per[lf]), t1 - t0, C), dtype=torch.complex128, device=dev)
                for k, d in enumerate(dd):
                    n0, fse, poly, m0 = delays[d]
                    up = lambda v: torch.from_numpy(np.ascontiguousarray(v[t0:t1])).to(dev)[:, None]   # noqa: E731
                    s = up(n0) + ns
                    ok = good[k][s // spf]
                    w = ok.double().mean(dim=1)
                    weights[d][t0:t1] = w.cpu().numpy()
                    if order:
                        x = ns.double() / L
                        rot = _turn(-fr.freq_mhz * (up(poly[0]) * x * x + up(poly[1]) * x + up(poly[2])))
                    e = up(fse)
                    chan = (cs - C if fr.lsb and not d0.complex_sampling else cs) * fr.bw_mhz / C
                    ph = _turn(chan * e - (0 if order else fr.freq_mhz * up(poly[2])))
                    for m, b in enumerate(per[lf]):
                        if d0.nbits == 2:
                            q = s * nb + b
                            x = lut[d0.format][((loads[k][q >> 2] >> (2 * (q & 3)).to(torch.uint8)) & 3).long()] * ok
                        elif d0.complex_sampling:
                            q = 2 * (s * nb + b)
                            x = torch.complex(lut8[loads[k][q].long()], lut8[loads[k][q + 1].long()]) * ok
                        else:
                            x = lut8[loads[k][s * nb + b].long()] * ok
                        if side:
                            nt = tones[d, b].numel()
                            tones[d, b].index_add_(0, ((s + m0) % nt).reshape(-1), x.reshape(-1))
                        F = torch.fft.fft(x * rot if order else x.to(torch.complex128), dim=1)
                        F = (F[:, C:] if fr.lsb and not d0.complex_sampling else F[:, :C]) * ph
                        X[k * len(per[lf]) + m] = F
                        if side:
                            p = F.real ** 2 + F.imag ** 2
                            kurt[d, b] += torch.stack([p.sum(0), (p * p).sum(0)])
                A = X.permute(2, 0, 1).contiguous()
                V[fl, lf] += torch.bmm(A, A.conj().permute(0, 2, 1).contiguous())
                del X, A

    def source(d, b):
        """Recorded band and first channel of a band (zoom bands are windows of their parents)."""
        ds = cfg.datastreams[d]
        if b < len(ds.recbands):
            return b, 0
        lz, pol = ds.zoombands[b - len(ds.recbands)]
        _, parent, off = ds.zoomfreqs[lz]
        return ds.recbands.index((parent, pol)), off

    def product(d1, b1, d2, b2, n):
        (r1, c1), (r2, c2) = source(d1, b1), source(d2, b2)
        (fl, lf, i), (_, _, j) = rows[d1, r1], rows[d2, r2]
        return V[fl, lf][c1:c1 + n, i, j]

    nprod = max(len(p) for b in cfg.baselines for _, p in b.freqs)
    bpa = 2 if nprod > 2 else 1
    parts = []
    for fi, fr in enumerate(cfg.freqs):
        for bl in cfg.baselines:
            for f, prods in bl.freqs:
                if f == fi:
                    parts += [product(bl.ds1, b1, bl.ds2, b2, fr.nchan) for b1, b2 in prods]

    def words(vals):
        v = np.zeros(len(vals) + len(vals) % 2)
        v[: len(vals)] = vals
        return torch.from_numpy(v).view(torch.complex128).to(dev)

    for fi in range(len(cfg.freqs)):
        for bl in cfg.baselines:
            for f, prods in bl.freqs:
                if f == fi:
                    parts.append(words([float(np.sum(weights[bl.ds1] * weights[bl.ds2]))] * len(prods)))

    def bands(d):
        ds = cfg.datastreams[d]
        for b in range(len(ds.recbands) + len(ds.zoombands)):
            rec, _ = source(d, b)
            fi = ds.recfreqs[ds.recbands[b][0]] if b < len(ds.recbands) else ds.zoomfreqs[ds.zoombands[b - len(ds.recbands)][0]][0]
            mate = [x for x, (lf, _) in enumerate(ds.recbands) if lf == ds.recbands[rec][0] and x != rec]
            yield b, rec, fi, (mate[0] if mate else None)

    for d in range(nds):
        for w in range(bpa):
            for b, rec, fi, mate in bands(d):
                n = cfg.freqs[fi].nchan
                _, off = source(d, b)
                other = rec if w == 0 else mate
                fl, lf, i = rows[d, rec]
                v = V[fl, lf][off:off + n, i, rows[d, other][2]].clone() if other is not None else torch.zeros(n, dtype=torch.complex128, device=dev)
                parts.append(v)
    for d in range(nds):
        vals = [float(np.sum(weights[d])) if w == 0 or mate is not None else 0.0 for w in range(bpa) for _, _, _, mate in bands(d)]
        parts.append(words(vals))
    if side:
        for d, ds in enumerate(cfg.datastreams):
            for b in range(len(ds.recbands)):
                nt = tones[d, b].numel() // 2                         # 1 MHz comb: tone k at k + 1 MHz
                z = torch.fft.fft(torch.complex(tones[d, b], torch.zeros_like(tones[d, b])))
                parts.append(z[1:nt + 1].clone())
    res = torch.cat([p.reshape(-1) for p in parts])
    if not side:
        return res.cpu().numpy() if case.get("host") else res
    sk = []
    for d, ds in enumerate(cfg.datastreams):
        for b in range(len(ds.recbands)):
            s1, s2 = kurt[d, b]
            sk.append(((B * s2 / (s1 * s1) - 1) * B / (B - 1) - 1).cpu().numpy())
    return {"results": res, "kurtosis": np.stack(sk)}


def exact(case, seed):
    if case["kind"] == "mux":
        return None                                  # bytes: compared as they are
    return _exact_subint(case, seed)
