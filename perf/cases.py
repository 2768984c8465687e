"""The calls whose speed is tracked: what each is, its inputs, one pass, the
work it cannot avoid, and its result in 64 bits.

A case is a dict of plain values; its "kind" names the operator:

  channelizer  MultiRateChannelizer on device buffers, channels with and
               without discriminator tails, batched and per-channel form
  serving      Server: a burst of chunks of several streams from host memory
  resampler    PolyphaseResampler on device buffers
  shift        FreqShift with one or more shifts, float or int16 samples
  receiver     the 16-bit narrow-band receiver: shift, FIR, discriminator, all
               on complex int16 device buffers
  fir          FirFilter with complex taps
  fir_bank     FirBank: one real-tap filter per channel
  iir          IirFilter, one stream
  iir_bank     IirBank, many exact streams
  fm           FmDemodulator on host arrays, samples in, audio out

Streams carry their state from pass to pass, as a program that feeds one
chunk after another has it; prepare() gives a fresh stream.
"""
import cmath
import ctypes
import math
import random

import numpy as np
import torch

import libfalcon_dsp_amd as fd
from libfalcon_dsp_amd._native import check
from libfalcon_dsp_amd.signals import kaiser_sinc
from libfalcon_dsp_amd.workloads import RATES, channel

# output rates off the input rate's divisors (up 2 to 48), beside the plain ones
FINE_RATES = [48_000, 192_000, 400_000, 1_600_000, 3_000_000, 12_500, 250_000, 2_500_000]
# resampling ratios in the tests and in audio and radio use
RATIOS = [(1, 2), (2, 3), (3, 2), (4, 5), (5, 2), (5, 1), (2, 9), (1, 8), (1, 80), (160, 147)]


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # a 20 Msps recording cut into 32 channels, 0.84 s at once
        dict(name="chan32_recording", kind="channelizer", fs=20_000_000, n=1 << 24, channels=32, plan=2, rates="plain",
             tails=0.0, per_up=32, batched=True),
        # one live chunk (0.8 ms) of a small receiver with rational rates and an FM channel
        dict(name="chan7_live_chunk", kind="channelizer", fs=20_000_000, n=16_411, channels=7, plan=1, rates="fine",
             tails=0.15, per_up=32, batched=True),
        # an FM scanner: 16 stations' angles from 0.1 s of a 20 Msps band
        dict(name="fm_scanner16", kind="channelizer", fs=20_000_000, n=2_097_189, channels=16, plan=3, rates="plain",
             tails=1.0, per_up=64, batched=True),
        # a server that gets one chunk from each of 24 clients at about the same time
        dict(name="serving_burst24", kind="serving", fs=25_000_000, streams=24, chunk=65_536, plan=5, rounds=1),
        # one live chunk of one stream to 4/5 of its rate
        dict(name="resample_chunk", kind="resampler", up=4, down=5, per_phase=24, n=65_536),
        # 16 receivers' basebands from one recording
        dict(name="shift16_recording", kind="shift", fs=25_000_000, shifts=16, n=1 << 22, sample="cf32"),
        # a 16-bit radio front end's chunk down to FM angles
        dict(name="receiver16_chunk", kind="receiver", fs=25_000_000, taps=64, n=1 << 18),
        # an equaliser or matched filter over a second of 1 Msps signal
        dict(name="fir129_stream", kind="fir", taps=129, n=1_000_003, sample="cf32"),
        # the same kind of filter on each of 256 sensor channels
        dict(name="fir_bank256", kind="fir_bank", channels=256, taps=512, n=1 << 17),
        # a recursive low-pass over a long stream
        dict(name="iir4_stream", kind="iir", order=4, cutoff=0.2, n=1 << 20, sample="cf32"),
        # the same low-pass on 1024 streams, each as a sequential filter gives it
        dict(name="iir4_bank1024", kind="iir_bank", order=4, cutoff=0.2, streams=1024, n=8192, sample="cf32"),
        # broadcast FM to audio, host arrays in and out
        dict(name="fm_audio_chunk", kind="fm", offset=-200_000, tau_us=75, n=1 << 18),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["channelizer", "channelizer", "channelizer", "serving", "resampler", "resampler", "shift",
                       "receiver", "fir", "fir", "fir_bank", "iir", "iir_bank", "fm"])
    if kind == "channelizer":
        tails = rng.choice([0.0, 0.0, 0.25, 1.0])
        rates = rng.choice(["plain", "plain", "fine"])
        batched = tails > 0 or rng.random() < 0.8
        chans = _log(rng, 1, 16 if tails == 1.0 else 32)
        # the per-channel form writes a full-rate copy per channel: shorter chunks
        n = _log(rng, 1 << 12, (1 << 24 if rates == "plain" and tails < 1.0 else 1 << 22) if batched else (1 << 21))
        return dict(kind=kind, fs=rng.choice([20_000_000, 25_000_000]), n=n, channels=chans,
                    plan=rng.randrange(1 << 20), rates=rates, tails=tails,
                    per_up=64 if tails == 1.0 else rng.choice([32, 32, 32, 48] if tails else [32, 32, 32, 16, 48]),
                    batched=batched)
    if kind == "serving":
        return dict(kind=kind, fs=25_000_000, streams=_log(rng, 2, 24), chunk=_log(rng, 1 << 12, 1 << 16),
                    plan=rng.randrange(1 << 20), rounds=rng.choice([1, 2]))
    if kind == "resampler":
        up, down = rng.choice(RATIOS)
        return dict(kind=kind, up=up, down=down, per_phase=rng.choice([8, 16, 24, 32, 33, 64]),
                    n=_log(rng, 1 << 12, (1 << 23) // up if up > 1 else 1 << 23))
    if kind == "shift":
        k = _log(rng, 1, 16)
        return dict(kind=kind, fs=rng.choice([20_000_000, 25_000_000]), shifts=k, n=_log(rng, 1 << 12, (1 << 26) // max(k, 8)),
                    sample=rng.choice(["cf32", "cf32", "ci16"]))
    if kind == "receiver":
        return dict(kind=kind, fs=rng.choice([20_000_000, 25_000_000]), taps=_log(rng, 16, 256),
                    n=_log(rng, 1 << 12, 1 << 20))
    if kind == "fir":
        return dict(kind=kind, taps=_log(rng, 8, 512), n=_log(rng, 1 << 12, 1 << 22),
                    sample=rng.choice(["cf32", "cf32", "cf32", "ci16"]))
    if kind == "fir_bank":
        k = _log(rng, 4, 256)
        return dict(kind=kind, channels=k, taps=_log(rng, 16, 512), n=_log(rng, 1 << 10, (1 << 25) // max(k, 128)))
    if kind == "iir":
        sample = rng.choice(["cf32", "cf32", "f32", "ci16"])
        # int16 outputs of one stream run as one sequential wave: short chunks
        return dict(kind=kind, order=rng.choice([1, 2, 4, 6]), cutoff=round(rng.uniform(0.1, 0.5), 3),
                    n=_log(rng, 1 << 10, 1 << 14 if sample == "ci16" else 1 << 20), sample=sample)
    if kind == "iir_bank":
        s = _log(rng, 16, 1024)
        return dict(kind=kind, order=rng.choice([2, 4, 6]), cutoff=round(rng.uniform(0.1, 0.5), 3), streams=s,
                    n=_log(rng, 256, 8192), sample=rng.choice(["cf32", "cf32", "ci16"]))
    return dict(kind="fm", offset=rng.choice([-250_000, -200_000, 150_000, 300_000]), tau_us=rng.choice([75, 50]),
                n=_log(rng, 1 << 13, 1 << 18))


# ---------------------------------------------------------------------------
# inputs and plans
# ---------------------------------------------------------------------------
_STREAM = []


def _stream():
    """the program's one HIP stream"""
    if not _STREAM:
        _STREAM.append(fd.Stream())
    return _STREAM[0]


class _Buffer:
    """A torch tensor as the library's device buffer (the part of DeviceBuffer that the operators read)."""

    def __init__(self, t, count=None):
        self.t, self.count = t, t.numel() if count is None else count
        self.ptr = ctypes.c_void_p(t.data_ptr())

    def at(self, offset):
        return ctypes.c_void_p(self.ptr.value + offset * self.t.element_size())


def _ci16_buffer(t):
    """(..., 2) int16 samples: the count is in pairs"""
    b = _Buffer(t, t.numel() // 2)
    b.at = lambda offset: ctypes.c_void_p(t.data_ptr() + 4 * offset)
    return b


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _noise(g, *shape, scale=1.0):
    """complex white noise of power scale^2"""
    t = torch.randn(*shape, 2, generator=g, device="cuda") * (scale / math.sqrt(2))
    return torch.view_as_complex(t)


def _tone(n, rev, device="cuda"):
    """e^{j 2 pi rev k}, k < n, the phase in 64 bits"""
    k = torch.arange(n, dtype=torch.float64, device=device)
    return torch.polar(torch.ones_like(k), 2 * math.pi * torch.remainder(k * rev, 1.0))


def _fm(n, fs, carrier, g, deviation=75e3):
    """a broadcast-like FM carrier: three audio tones of random pitch, the phase their integral in closed form"""
    k = torch.arange(n, dtype=torch.float64, device="cuda")
    f = (300 + 2700 * torch.rand(3, generator=g, device="cuda", dtype=torch.float64)).tolist()
    ph = torch.remainder(k * (carrier / fs), 1.0)
    for v in f:
        ph += deviation / (3 * 2 * math.pi * v) * torch.sin(2 * math.pi * (v / fs) * k)
    return torch.polar(torch.ones_like(ph), 2 * math.pi * torch.remainder(ph, 1.0))


def _channels(case):
    """the channel set of a channelizer case: a function of the case alone"""
    r, fs = random.Random(case["plan"]), case["fs"]
    rates = RATES if case["rates"] == "plain" else FINE_RATES
    # stations lie far enough apart for the filters to separate them (about 2.8 / taps of the rate)
    step = 0.055 if case["per_up"] >= 64 else 0.1
    stations = [k * step for k in range(-int(0.46 / step), int(0.46 / step) + 1) if k]
    r.shuffle(stations)
    out = []
    for _ in range(case["channels"]):
        tail = r.random() < case["tails"] and bool(stations)
        at = stations.pop() + r.uniform(-0.002, 0.002) if tail else r.uniform(-0.45, 0.45)
        out.append(channel(fs, int(round(at * fs)) or 1, 250_000 if tail else r.choice(rates),
                           taps_per_up=case["per_up"], tail="discriminator" if tail else None))
    return out


def _band(case, seed):
    """noise plus a carrier in each channel's pass band: a tone, weak beside the FM stations that
    channels with a discriminator tail listen to"""
    n, fs, g = case["n"], case["fs"], _gen(seed)
    weak = 0.02 if case["tails"] else 1.0
    x = _noise(g, n, scale=weak)
    for c in _channels(case):
        off = (torch.rand(1, generator=g, device="cuda").item() - 0.5) * 0.5 * c["output_sample_rate_in_sps"]
        if c.get("tail"):
            x += _fm(n, fs, -c["freq_shift_in_hz"], g).to(torch.complex64)
        else:
            x += (weak * _tone(n, (-c["freq_shift_in_hz"] + off) / fs)).to(torch.complex64)
    return x


def _shifts(case):
    k, fs = case["shifts"], case["fs"]
    return [int(round(0.4 * fs * (-1 + 2 * i / max(k - 1, 1)))) or 1_234_567 for i in range(k)]


def _to_i16(x, scale):
    """samples of a 16-bit front end"""
    return torch.view_as_real(x * scale).round().clamp(-32768, 32767).to(torch.int16).contiguous()


def _fir_taps(m):
    """a complex band-pass: a windowed sinc around 0.13 cycles a sample"""
    h = kaiser_sinc(m, 0.1, 8.0).astype(np.complex128) * np.exp(2j * np.pi * 0.13 * np.arange(m))
    return h.astype(np.complex64)


def _bank_taps(case):
    r = random.Random(case["channels"] * 4096 + case["taps"])
    return np.stack([kaiser_sinc(case["taps"], r.uniform(0.05, 0.45), 8.0) for _ in range(case["channels"])])


def _butter(order, cutoff):
    """Butterworth low-pass, cutoff in parts of Nyquist, by the bilinear transform: (b, a) as float32 values"""
    w = 2 * math.tan(math.pi * cutoff / 2)
    poles = [w * cmath.exp(1j * math.pi * (2 * k + order + 1) / (2 * order)) for k in range(order)]
    z = [(2 + p) / (2 - p) for p in poles]
    a = np.real(np.poly(z))
    b = np.real(np.poly([-1.0] * order))
    b = b * a.sum() / b.sum()
    return b.astype(np.float32), a.astype(np.float32)


def _serving_plan(case):
    """(streams' channels, [(stream, first sample, samples)]): chunks of a quarter of the largest up to it"""
    r, fs = random.Random(case["plan"]), case["fs"]
    chans, reqs, at = [], [], [0] * case["streams"]
    for s in range(case["streams"]):
        fm = r.random() < 0.25
        f = int(round(-10e6 + r.randrange(16) * 20e6 / 15)) or 1
        chans.append(channel(fs, f, 250_000 if fm else r.choice(RATES), tail="discriminator" if fm else None))
    for _ in range(case["rounds"]):
        for s in range(case["streams"]):
            n = r.randrange(case["chunk"] // 4, case["chunk"] + 1)
            reqs.append((s, at[s], n))
            at[s] += n
    return chans, reqs, at


def _serving_inputs(case, seed):
    chans, _, total = _serving_plan(case)
    g, fs, out = _gen(seed), case["fs"], []
    for c, n in zip(chans, total):
        x = _noise(g, n, scale=0.1).to(torch.complex64)
        if c.get("tail"):
            x += _fm(n, fs, -c["freq_shift_in_hz"], g).to(torch.complex64)
        out.append(x)
    return out


def _fm_input(case, seed):
    g = _gen(seed)
    x = _fm(case["n"], 1_140_000, -case["offset"], g) + _noise(g, case["n"], scale=0.02)
    return x.to(torch.complex64)


def _inputs(case, seed):
    """the device tensor(s) a case's stream reads"""
    kind = case["kind"]
    if kind == "channelizer":
        return _band(case, seed)
    if kind == "serving":
        return _serving_inputs(case, seed)
    if kind == "fm":
        return _fm_input(case, seed)
    g, n = _gen(seed), case["n"]
    if kind == "receiver":
        x = _fm(n, case["fs"], 3_000_000, g, deviation=200e3) + _noise(g, n, scale=0.02)
        return _to_i16(x, 12_000.0)
    if kind == "fir_bank":
        return _noise(g, case["channels"], n)
    if kind == "iir_bank":
        x = _noise(g, case["streams"], n)
    else:
        x = _noise(g, n)
    if kind == "resampler":
        x += _tone(n, 0.1).to(torch.complex64)
    if case.get("sample") == "ci16":
        return _to_i16(x, 4096.0)
    if case.get("sample") == "f32":
        return x.real.contiguous()
    return x


def prepare(case, seed):
    kind = case["kind"]
    x = _inputs(case, seed)
    s = dict(kind=kind, x=x, stream=_stream(), sample=case.get("sample"), n=case.get("n"))
    if kind == "channelizer":
        chans = _channels(case)
        h = fd.MultiRateChannelizer(case["fs"], chans, batched=case["batched"])
        s["outs"] = [torch.zeros(m + 1, dtype=torch.float32 if c.get("tail") else torch.complex64, device="cuda")
                     for m, c in zip(h.max_out(case["n"]), chans)]
        s.update(h=h, d_in=_Buffer(x), d_outs=[_Buffer(t) for t in s["outs"]])
    elif kind == "serving":
        chans, reqs, _ = _serving_plan(case)
        h = fd.Server(case["fs"], max_streams=case["streams"], max_chunk=1 << 18, max_batch=1 << 21,
                      state_bytes=64 << 20)
        host = [t.cpu().numpy() for t in x]
        ids = [h.admit(c) for c in chans]
        s.update(h=h, x=None, reqs=[(ids[k], host[k][p:p + m].copy()) for k, p, m in reqs])
    elif kind == "resampler":
        taps = kaiser_sinc(case["per_phase"] * case["up"], 0.5 / max(case["up"], case["down"]), 8.0, gain=case["up"])
        h = fd.PolyphaseResampler(case["up"], case["down"], taps.astype(np.complex64))
        s["out"] = torch.zeros(-(-case["n"] * case["up"] // case["down"]) + 1, dtype=torch.complex64, device="cuda")
        s.update(h=h, d_in=_Buffer(x), d_out=_Buffer(s["out"]))
    elif kind == "shift":
        k = case["shifts"]
        s["h"] = fd.FreqShift(case["fs"], _shifts(case))
        if case["sample"] == "ci16":
            s["out"] = torch.zeros(k, case["n"], 2, dtype=torch.int16, device="cuda")
            s.update(d_in=_ci16_buffer(x), d_out=_ci16_buffer(s["out"]))
        else:
            s["out"] = torch.zeros(k, case["n"], dtype=torch.complex64, device="cuda")
            s.update(d_in=_Buffer(x), d_out=_Buffer(s["out"]))
    elif kind == "receiver":
        s.update(shift=fd.FreqShift(case["fs"], -3_000_000), disc=fd.PolarDiscriminator(),
                 fir=fd.FirFilter(kaiser_sinc(case["taps"], 0.02, 8.0).astype(np.complex64)))
        s["mid"], s["low"] = torch.zeros_like(x), torch.zeros_like(x)
        s["out"] = torch.zeros(case["n"], dtype=torch.float32, device="cuda")
        s.update(d_in=_ci16_buffer(x), d_mid=_ci16_buffer(s["mid"]), d_low=_ci16_buffer(s["low"]),
                 d_out=_Buffer(s["out"]))
    elif kind == "fir":
        s["out"] = torch.zeros_like(x)
        buf = _ci16_buffer if case["sample"] == "ci16" else _Buffer
        s.update(h=fd.FirFilter(_fir_taps(case["taps"])), d_in=buf(x), d_out=buf(s["out"]))
    elif kind == "fir_bank":
        s["out"] = torch.zeros_like(x)
        s.update(h=fd.FirBank(_bank_taps(case)), d_in=_Buffer(x), d_out=_Buffer(s["out"]))
    elif kind in ("iir", "iir_bank"):
        b, a = _butter(case["order"], case["cutoff"])
        s["out"] = torch.zeros_like(x)
        buf = _ci16_buffer if case["sample"] == "ci16" else _Buffer
        h = fd.IirFilter(b, a) if kind == "iir" else fd.IirBank(b, a, case["streams"])
        s.update(h=h, d_in=buf(x), d_out=buf(s["out"]))
    else:
        s.update(h=fd.FmDemodulator(1_140_000, case["offset"], tau=case["tau_us"] * 1e-6), x=x.cpu().numpy())
    torch.cuda.synchronize()
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(s):
    kind, st, n = s["kind"], s["stream"], s["n"]
    if kind == "channelizer":
        counts = s["h"].apply_device(s["d_in"], n, s["d_outs"], st)
        return [t[:k] for t, k in zip(s["outs"], counts)]
    if kind == "serving":
        h = s["h"]
        tickets = [h.submit(sid, x) for sid, x in s["reqs"]]
        return [h.result(t)[0] for t in tickets]
    if kind == "resampler":
        return s["out"][:s["h"].apply_device(s["d_in"], n, s["d_out"], st)]
    if kind == "shift":
        f = s["h"].apply_ci16_device if s["sample"] == "ci16" else s["h"].apply_device
        f(s["d_in"], n, s["d_out"], n, st)
        return s["out"]
    if kind == "receiver":
        s["shift"].apply_ci16_device(s["d_in"], n, s["d_mid"], n, st)
        s["fir"].apply_ci16_device(s["d_mid"], n, s["d_low"], st)
        got = ctypes.c_size_t()
        check(fd.lib().fdsp_discriminator_apply_ci16_device(s["disc"].h, s["d_low"].ptr, n, s["d_out"].ptr,
                                                            ctypes.byref(got), st.h))
        return {"low": s["low"], "angle": s["out"][:got.value]}
    if kind == "fir":
        f = s["h"].apply_ci16_device if s["sample"] == "ci16" else s["h"].apply_device
        f(s["d_in"], n, s["d_out"], st)
        return s["out"]
    if kind == "fir_bank":
        s["h"].apply_device(s["d_in"], n, n, s["d_out"], n, st)
        return s["out"]
    if kind == "iir":
        s["h"].apply_device(s["d_in"], n, s["d_out"], st, kind=s["sample"])
        return s["out"]
    if kind == "iir_bank":
        s["h"].apply_device(s["d_in"], n, n, s["d_out"], n, st, ci16=s["sample"] == "ci16")
        return s["out"]
    pcm, audio = s["h"].demod_mono(s["x"], audio=True)
    return {"pcm": pcm, "audio": audio}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _chan_work(chans, n):
    """(output bytes, flops) of n inputs through a channel set: a complex tap costs 8 flops, an angle about 30"""
    size = flops = 0
    for c in chans:
        k = n * c["up_rate"] / c["down_rate"]
        size += k * (4 if c.get("tail") else 8)
        flops += k * (8 * len(c["taps"]) / c["up_rate"] + (30 if c.get("tail") else 0))
    return size, flops


def work(case):
    kind, n = case["kind"], case.get("n")
    if kind == "channelizer":
        size, flops = _chan_work(_channels(case), n)
        return dict(bytes=8 * n + size, flops=flops)
    if kind == "serving":
        chans, reqs, _ = _serving_plan(case)
        size = flops = 0
        for s, _, m in reqs:
            b, f = _chan_work([chans[s]], m)
            size, flops = size + 8 * m + b, flops + f
        return dict(bytes=size, flops=flops)
    if kind == "resampler":
        k = n * case["up"] / case["down"]
        return dict(bytes=8 * (n + k), flops=4 * case["per_phase"] * k)
    if kind == "shift":
        size = 4 if case["sample"] == "ci16" else 8
        return dict(bytes=size * n * (1 + case["shifts"]), flops=12 * n * case["shifts"])
    if kind == "receiver":
        # int16 in, the low-passed samples and the angles out
        return dict(bytes=12 * n, flops=n * (12 + 8 * case["taps"] + 30))
    if kind == "fir":
        return dict(bytes=(8 if case["sample"] == "ci16" else 16) * n, flops=8 * case["taps"] * n)
    if kind == "fir_bank":
        k = n * case["channels"]
        return dict(bytes=16 * k, flops=4 * case["taps"] * k)
    if kind in ("iir", "iir_bank"):
        k = n * case.get("streams", 1)
        parts = 1 if case["sample"] == "f32" else 2
        size = {"cf32": 16, "f32": 8, "ci16": 8}[case["sample"]]
        return dict(bytes=size * k, flops=parts * 2 * (2 * case["order"] + 1) * k)
    # two 64-tap decimators by 5, one angle and one recurrence step between them
    return dict(bytes=8 * n + 6 * n / 25, flops=n / 5 * (8 * 64 + 40) + n / 25 * 4 * 64)


def tolerance(case):
    """32-bit sums of up to 512 products: about 1e-6 of the result, four times what another order of sums shows.
    Whole numbers follow the sequential arithmetic exactly, but for the audio, whose truncation turns a last-bit
    difference of the float sample into a step now and then."""
    kind = case["kind"]
    if kind == "receiver":
        return dict(rel=2e-6, max=2e-5, differ=0.0)
    if kind == "fm":
        return dict(rel=4e-6, max=4e-5, differ=0.01)
    if kind == "iir_bank" or case.get("sample") == "ci16":
        return "exact"  # the sequential filter's outputs, bit for bit
    if kind == "iir":
        return dict(rel=1e-5, max=1e-4)
    if kind in ("channelizer", "serving"):
        # angles: the error of a sample over its own size, which in a filter's first outputs is small
        return dict(rel=4e-6, max=4e-3) if case.get("tails", 1) else dict(rel=2e-6, max=2e-5)
    return dict(rel=2e-6, max=2e-5)


# ---------------------------------------------------------------------------
# the same in 64 bits, from a fresh stream
# ---------------------------------------------------------------------------
def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _shift64(x, fs, f):
    """x[n] e^{j 2 pi (f/fs) (n mod R)}, R the period fs/|f| scaled by ten until it is 1e5 or more, rounded"""
    r = fs / abs(f)
    while r < 1e5:
        r *= 10
    k = torch.remainder(torch.arange(x.numel(), dtype=torch.int64, device=x.device), int(math.floor(r + 0.5)))
    rev = torch.remainder(k.to(torch.float64) * (f / fs), 1.0)
    return x.to(torch.complex128) * torch.polar(torch.ones_like(rev), 2 * math.pi * rev)


def _resample64(x, up, down, taps):
    """outputs whose anchor floor(n down / up) lies in x, the real taps at phase (n down) mod up"""
    h = torch.from_numpy(np.real(taps).astype(np.float64)).to(x.device)
    per = -(-h.numel() // up)
    h = torch.cat([h, h.new_zeros(per * up - h.numel())])
    n = torch.arange(-(-x.numel() * up // down), dtype=torch.int64, device=x.device) * down
    at, ph = torch.div(n, up, rounding_mode="floor"), torch.remainder(n, up)
    xp = torch.cat([x.new_zeros(per - 1), x])
    y = torch.zeros(n.numel(), dtype=x.dtype, device=x.device)
    for j in range(per):
        y += h[j * up + ph] * xp[at + (per - 1 - j)]
    return y


def _angles64(y):
    return torch.angle(y[1:] * y[:-1].conj())


def _channel64(x, fs, c):
    y = _resample64(_shift64(x, fs, c["freq_shift_in_hz"]), c["up_rate"], c["down_rate"], c["taps"])
    return _angles64(y) if c.get("tail") else y


def _convolve64(x, h):
    """the first x.shape[-1] outputs of x * h along the last axis"""
    n = x.shape[-1]
    size = 1 << (n + h.shape[-1] - 1).bit_length()
    hf = torch.fft.fft(h.to(torch.complex128), size)
    return torch.fft.ifft(torch.fft.fft(x.to(torch.complex128), size) * hf)[..., :n]


def _impulse(b, a, length=4096):
    b, a = [float(v) for v in b], [float(v) for v in a]
    h = []
    for n in range(length):
        v = b[n] if n < len(b) else 0.0
        for j in range(1, min(len(a), n + 1)):
            v -= a[j] * h[n - j]
        h.append(v / a[0])
    return torch.tensor(h, dtype=torch.float64)


def exact(case, seed):
    kind = case["kind"]
    x = _inputs(case, seed)
    if kind == "channelizer":
        return [_channel64(x, case["fs"], c) for c in _channels(case)]
    if kind == "serving":
        chans, reqs, _ = _serving_plan(case)
        whole = [_channel64(t, case["fs"], c) for t, c in zip(x, chans)]
        done, out = [0] * len(chans), []
        for s, p, m in reqs:
            c = chans[s]
            end = -(-(p + m) * c["up_rate"] // c["down_rate"]) - (1 if c.get("tail") else 0)
            out.append(whole[s][done[s]:max(end, done[s])].cpu().numpy())
            done[s] = max(end, done[s])
        return out
    if kind == "resampler":
        taps = kaiser_sinc(case["per_phase"] * case["up"], 0.5 / max(case["up"], case["down"]), 8.0, gain=case["up"])
        return _resample64(x.to(torch.complex128), case["up"], case["down"], taps)
    if kind == "shift":
        if case["sample"] == "ci16":
            return None
        return torch.stack([_shift64(x, case["fs"], f) for f in _shifts(case)])
    if kind == "receiver":
        return None  # angles of whole numbers: while the filter fills they are 0 and 1, and one step turns an angle
    if kind in ("fir", "iir", "iir_bank") and case["sample"] == "ci16":
        return None
    if kind == "fir":
        return _convolve64(x, torch.from_numpy(_fir_taps(case["taps"]).astype(np.complex128)).to(x.device))
    if kind == "fir_bank":
        h = torch.from_numpy(_bank_taps(case).astype(np.float64)).to(x.device)
        return torch.cat([_convolve64(x[k:k + 16], h[k:k + 16]) for k in range(0, x.shape[0], 16)])
    if kind in ("iir", "iir_bank"):
        y = _convolve64(x, _impulse(*_butter(case["order"], case["cutoff"])).to(x.device))
        return y.real.contiguous() if case["sample"] == "f32" else y
    # FM: shift, decimate, angle, de-emphasis (x = exp(-1 / (200000 tau))), decimate
    up, down, iso = fd.resample_fir_params(1_140_000, 228_000)
    y = _angles64(_resample64(_shift64(x, 1_140_000, case["offset"]), up, down, iso))
    p = math.exp(-1.0 / (200_000.0 * case["tau_us"] * 1e-6))
    y = _convolve64(y, _impulse([np.float32(1 - p)], [1.0, np.float32(-p)]).to(y.device)).real
    up, down, mono = fd.resample_fir_params(228_000, 45_600)
    return {"pcm": None, "audio": _resample64(y, up, down, mono).cpu().numpy()}
