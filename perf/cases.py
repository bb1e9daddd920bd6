"""Performance cases of the audio library: what its users run, through its public entry points.

A case is a dict of plain values; `kind` names the path and the other fields its sizes and options.
Clips are ragged: a case fixes the set of lengths (spread evenly over the logarithm of
[min_s, max_s]), the seed decides which clip gets which and what the clips hold.

  logmel    the whole chain in one launch (rppt_logmel_fused_gpu)
  chain     the four drop-in calls: pre-emphasis, spectrogram, mel filter bank, to_decibels
  dbspec    spectrogram and to_decibels without a mel bank, as a viewer or a CNN on spectra runs them
  packed    the launch one served batch runs: clips back to back, dense dB blocks per clip
  front     interleaved stereo at 48 kHz down-mixed, resampled and turned into log-mel in one call
  resample  the two drop-in calls in front of feature extraction: down-mixing, then resampling
  trim      non-silent region detection, then the fused launch on the regions it reports
"""
import math
import random

import numpy as np
import torch

from rpp_amd import api, synth

SPEECH = dict(rate=16000, nfft=512, window=400, hop=160, mels=80)
MUSIC = dict(rate=44100, nfft=1024, window=1024, hop=256, mels=128)


def listed():
    return [
        # one short utterance: a single request answered as it comes, where only latency counts
        dict(name="logmel_one_clip", kind="logmel", clips=1, min_s=2.0, max_s=2.0, precision="fp16x3", ref=1.0, **SPEECH),
        # a small training or evaluation batch of 1-3 s clips through the drop-in calls
        dict(name="chain_batch8", kind="chain", clips=8, min_s=1.0, max_s=3.0, **SPEECH),
        # the drop-in calls over a data loader's batch of ragged utterances
        dict(name="chain_batch128", kind="chain", clips=128, min_s=0.5, max_s=20.0, **SPEECH),
        # feature extraction over a corpus: a big ragged batch in one launch
        dict(name="logmel_batch512", kind="logmel", clips=512, min_s=0.5, max_s=20.0, precision="fp16x3", ref=1.0, **SPEECH),
        # the same for music
        dict(name="logmel_music256", kind="logmel", clips=256, min_s=2.0, max_s=10.0, precision="fp16x3", ref=1.0, **MUSIC),
        # a front end of other dimensions (frames of 512 every 128 samples, 40 filters), bf16 split products
        dict(name="logmel_hop128_bf16x3", kind="logmel", clips=96, min_s=0.7, max_s=12.0, precision="bf16x3", ref=1.0,
             rate=16000, nfft=512, window=512, hop=128, mels=40),
        # plain FP32 arithmetic with every clip's maximum as the dB reference
        dict(name="logmel_fp32_clipref", kind="logmel", clips=64, min_s=0.5, max_s=20.0, precision="fp32", ref=0.0, **SPEECH),
        # magnitude spectra in dB below each recording's maximum
        dict(name="dbspec_2048", kind="dbspec", clips=12, min_s=5.0, max_s=30.0, rate=44100, nfft=2048, window=2048, hop=512,
             power=1),
        # one batch of the server: requests of very uneven length
        dict(name="packed_serve64", kind="packed", clips=64, min_s=0.25, max_s=30.0, precision="fp16x3", ref=1.0, **SPEECH),
        # studio recordings at 48 kHz, stereo, straight to 16 kHz speech features
        dict(name="front_stereo48k", kind="front", clips=48, min_s=20.0, max_s=60.0, precision="fp16x3", ref=1.0, in_rate=48000,
             channels=2, **SPEECH),
        # CD-rate stereo brought to 16 kHz mono by the two drop-in calls (a ratio that is no whole number)
        dict(name="resample_44k_stereo", kind="resample", clips=32, min_s=3.0, max_s=15.0, in_rate=44100, out_rate=16000,
             channels=2),
        # utterances with silence around them, trimmed before their features are taken
        dict(name="trim_batch256", kind="trim", clips=256, min_s=0.5, max_s=20.0, precision="fp16x3", ref=1.0, **SPEECH),
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["logmel", "logmel", "logmel", "chain", "chain", "dbspec", "packed", "front", "resample", "trim"])
    lo = _log_uniform(rng, 0.25, 6.0)
    hi = round(lo * _log_uniform(rng, 1.0, 16.0), 3)
    lo = round(lo, 3)
    mean = (lo + hi) / 2

    def clips(seconds):   # a batch whose total stays within `seconds` of audio
        return max(1, min(512, int(round(_log_uniform(rng, 1.0, max(1.5, min(512.0, seconds / mean)))))))

    def features(choices):
        rate, nfft, window, hop, mels = rng.choice(choices)
        return dict(rate=rate, nfft=nfft, window=window, hop=hop, mels=mels)

    speech = [(16000, 512, 400, 160, 80), (16000, 512, 400, 160, 64), (16000, 512, 320, 160, 80)]
    music = [(44100, 1024, 1024, 256, 128), (22050, 1024, 1024, 256, 80)]
    other = [(16000, 512, 512, 128, 40), (8000, 256, 200, 80, 40), (16000, 512, 400, 200, 80)]
    if kind == "logmel":
        precision = rng.choice(["fp16x3", "fp16x3", "bf16x3", "fp32"])
        total = 400.0 if precision == "fp32" else 1400.0
        return dict(kind=kind, clips=clips(total), min_s=lo, max_s=hi, precision=precision, ref=rng.choice([1.0, 1.0, 0.0]),
                    **features(speech + speech + music + other))
    if kind == "chain":
        return dict(kind=kind, clips=clips(400.0), min_s=lo, max_s=hi, **features(speech + music + other))
    if kind == "dbspec":
        rate, nfft, hop = rng.choice([(44100, 2048, 512), (22050, 1024, 256), (16000, 512, 160), (16000, 256, 64)])
        return dict(kind=kind, clips=clips(150.0), min_s=lo, max_s=hi, rate=rate, nfft=nfft, window=nfft - rng.choice([0, 0, 56]),
                    hop=hop, power=rng.choice([1, 2]))
    if kind == "packed":
        return dict(kind=kind, clips=clips(1000.0), min_s=lo, max_s=hi, precision="fp16x3", ref=1.0, **features(speech + other[:1]))
    if kind == "front":
        return dict(kind=kind, clips=clips(500.0), min_s=lo, max_s=hi, precision="fp16x3", ref=1.0,
                    in_rate=rng.choice([48000, 48000, 32000, 44100]), channels=2, **SPEECH)
    if kind == "resample":
        in_rate, out_rate = rng.choice([(44100, 16000), (48000, 16000), (22050, 16000), (8000, 16000), (48000, 44100)])
        return dict(kind=kind, clips=clips(250.0), min_s=lo, max_s=hi, in_rate=in_rate, out_rate=out_rate,
                    channels=rng.choice([1, 2, 2, 6]))
    return dict(kind="trim", clips=clips(1400.0), min_s=lo, max_s=hi, precision="fp16x3", ref=1.0, **features(speech))


# ------------------------------------------------------------------------------------------ sizes
LOBES, COEFFS = 16, 4091
OUT_16K = 16000


def _lengths(case):
    """The case's clip lengths in samples per channel, ascending."""
    n, rate = case["clips"], case.get("in_rate") or case["rate"]
    lo, hi = case["min_s"] * rate, case["max_s"] * rate
    return [max(1, int(round(lo * (hi / lo) ** ((i + 0.5) / n)))) for i in range(n)]


def _shuffled_lengths(case, seed):
    lengths = _lengths(case)
    random.Random(seed * 7919 + 17).shuffle(lengths)
    return np.array(lengths, np.int32)


def _out_length(n, in_rate, out_rate):
    return int(np.ceil(np.float32(n) * np.float32(out_rate) / np.float32(in_rate)))


def _stride(n):
    return n // 8 * 8 + 8


# ----------------------------------------------------------------------------------------- inputs
def _signal(gen, lengths, rate, stride, quiet_edges=False):
    """[clips][stride]: noise and a chirp per clip (with `quiet_edges` 80 dB down outside one burst), zero past its end."""
    n = len(lengths)
    L = torch.as_tensor(lengths, device="cuda", dtype=torch.float64).unsqueeze(1)
    r = torch.rand((4, n, 1), generator=gen, device="cuda", dtype=torch.float64)
    f0, f1 = 50 + r[0] * (rate / 4 - 50), 50 + r[1] * (rate / 2 - 50)
    x = torch.randn((n, stride), generator=gen, device="cuda") * 0.1
    step = max(1, (1 << 25) // stride)
    t = torch.arange(stride, device="cuda", dtype=torch.float64).unsqueeze(0)
    for i in range(0, n, step):
        s = slice(i, i + step)
        phase = (f0[s] + (f1[s] - f0[s]) * t / (2 * L[s])) * t / rate
        x[s] += 0.5 * torch.sin(2 * math.pi * (phase % 1.0)).float()
        if quiet_edges:
            a = (0.05 + 0.3 * r[2][s]) * L[s]
            b = (0.6 + 0.35 * r[3][s]) * L[s]
            x[s] *= torch.where((t >= a) & (t < b), 1.0, 1e-4).float()
        x[s] *= (t < L[s])
    return x


def _interleaved(gen, lengths, channels, stride):
    """[clips][stride * channels]: 16-bit samples scaled to [-1, 1), interleaved, zero past each clip's end."""
    n = len(lengths)
    x = torch.randint(-32768, 32768, (n, stride, channels), generator=gen, device="cuda", dtype=torch.int32).float() / 32768.0
    x *= (torch.arange(stride, device="cuda") < torch.as_tensor(lengths, device="cuda").unsqueeze(1)).unsqueeze(2)
    return x.reshape(n, stride * channels)


def _ints(a):
    return torch.as_tensor(np.ascontiguousarray(a, np.int32), device="cuda")


def _params(case):
    return api.logmel_params(nfft=case["nfft"], window_length=case["window"], window_step=case["hop"],
                             sample_rate=float(case["rate"]), max_freq=case["rate"] / 2.0, num_filter=case["mels"],
                             reference_magnitude=case.get("ref", 1.0))


def _inputs(case, seed):
    """(x, lengths) of a case: what the path is given, before any handle or buffer."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    lengths = _shuffled_lengths(case, seed)
    if case["kind"] in ("front", "resample"):
        return _interleaved(gen, lengths, case["channels"], _stride(int(lengths.max()))), lengths
    return _signal(gen, lengths, case["rate"], _stride(int(lengths.max())), case["kind"] == "trim"), lengths


def prepare(case, seed):
    kind = case["kind"]
    x, lengths = _inputs(case, seed)
    n = len(lengths)
    s = dict(case=case, x=x, handle=api.Handle(n), lengths=_ints(lengths))

    def zeros(*shape):
        return torch.zeros(shape, device="cuda")

    if kind in ("front", "resample"):
        lut, scale, center = synth.kaiser_sinc_lut(COEFFS, LOBES)
        s["sinc"] = api.make_window(torch.as_tensor(lut, device="cuda"), scale, center, LOBES, COEFFS)
        s["dims"] = _ints(np.stack([lengths, np.full(n, case["channels"])], 1).reshape(-1))
        out_rate = case["out_rate"] if kind == "resample" else OUT_16K
        longest = _out_length(int(lengths.max()), case["in_rate"], out_rate)
        if kind == "resample":
            s["mono"], s["res"] = zeros(n, _stride(int(lengths.max()))), zeros(n, _stride(longest))
            s["mono_dims"] = _ints(np.stack([lengths, np.ones(n)], 1).reshape(-1))
            s["in_rate"] = torch.full((n,), float(case["in_rate"]), device="cuda")
            s["out_rate"] = torch.full((n,), float(case["out_rate"]), device="cuda")
        else:
            s["params"], s["db"] = _params(case), zeros(n, case["mels"], longest // case["hop"] + 1)
        return s
    frames = lengths // case["hop"] + 1
    most, bins = int(frames.max()), case["nfft"] // 2 + 1
    if kind in ("chain", "dbspec"):
        rows = case["mels"] if kind == "chain" else bins
        s["spec"], s["db"] = zeros(n, bins, most), zeros(n, rows, most)
        s["db_dims"] = _ints(np.stack([frames, np.full(n, rows)], 1).reshape(-1))
        if kind == "chain":
            s["pre"], s["mel"] = torch.zeros_like(x), zeros(n, rows, most)
            s["coeffs"] = torch.full((n,), 0.97, device="cuda")
            s["mel_dims"] = _ints(np.stack([np.full(n, bins), frames], 1).reshape(-1))
        return s
    s["params"] = _params(case)
    if kind == "packed":
        s["src_off"] = torch.as_tensor(np.concatenate([[0], np.cumsum(lengths.astype(np.int64))[:-1]]), device="cuda")
        sizes = frames.astype(np.int64) * case["mels"]
        s["dst_off"] = torch.as_tensor(np.concatenate([[0], np.cumsum(sizes)[:-1]]), device="cuda")
        s["x"] = torch.cat([x[i, :int(l)] for i, l in enumerate(lengths)])
        s["db"] = zeros(int(sizes.sum()))
        return s
    s["db"] = zeros(n, case["mels"], most)
    if kind == "trim":
        s["begin"], s["count"] = torch.zeros_like(s["lengths"]), torch.zeros_like(s["lengths"])
    return s


def run(s):
    case, h = s["case"], s["handle"]
    kind = case["kind"]
    if kind == "logmel":
        api.logmel_fused(h, s["x"], s["db"], s["lengths"], s["params"], case["precision"])
        return s["db"]
    if kind == "chain":
        api.pre_emphasis_filter(h, s["x"], s["pre"], s["lengths"], s["coeffs"], "clamp")
        api.spectrogram(h, s["pre"], s["spec"], s["lengths"], nfft=case["nfft"], window_length=case["window"],
                        window_step=case["hop"])
        api.mel_filter_bank(h, s["spec"], s["mel"], s["mel_dims"], max_freq=case["rate"] / 2.0, num_filter=case["mels"],
                            sample_rate=float(case["rate"]))
        api.to_decibels(h, s["mel"], s["db"], s["db_dims"])
        return s["pre"], s["spec"], s["mel"], s["db"]
    if kind == "dbspec":
        api.spectrogram(h, s["x"], s["spec"], s["lengths"], nfft=case["nfft"], window_length=case["window"],
                        window_step=case["hop"], power=case["power"])
        api.to_decibels(h, s["spec"], s["db"], s["db_dims"], multiplier=20.0 if case["power"] == 1 else 10.0,
                        reference_magnitude=0.0)
        return s["spec"], s["db"]
    if kind == "packed":
        api.logmel_fused_packed(h, s["x"], s["src_off"], s["lengths"], s["db"], s["dst_off"], s["params"], case["precision"])
        return s["db"]
    if kind == "front":
        api.logmel_front_end(h, s["x"], s["db"], s["dims"], float(case["in_rate"]), float(OUT_16K), s["sinc"], s["params"],
                             case["precision"], channels=case["channels"])
        return s["db"]
    if kind == "resample":
        api.down_mixing(h, s["x"], s["mono"], s["dims"], channels=case["channels"])
        api.resample(h, s["mono"], s["res"], s["in_rate"], s["out_rate"], s["mono_dims"], s["sinc"])
        return s["mono"], s["res"]
    api.non_silent_region_detection(h, s["x"], s["lengths"], s["begin"], s["count"], -60.0, 2048, 0.0, 8192)
    api.logmel_fused_region(h, s["x"], s["db"], s["begin"], s["count"], s["params"], case["precision"])
    return s["begin"], s["count"], s["db"]


def work(case):
    """Samples read once, results written once; a real FFT per frame (2.5 N log2 N), 2 flops per non-zero mel weight."""
    kind, lengths = case["kind"], _lengths(case)
    if kind == "resample":
        out = sum(_out_length(n, case["in_rate"], case["out_rate"]) for n in lengths)
        return {"bytes": 4 * (sum(lengths) * (case["channels"] + 2) + out),
                "flops": 2 * case["channels"] * sum(lengths) + 4 * LOBES * out}
    taps = extra = 0
    if kind == "front":
        extra, lengths = 4 * case["channels"] * sum(lengths), [_out_length(n, case["in_rate"], OUT_16K) for n in lengths]
        taps = 4 * LOBES * sum(lengths)
    total, frames = sum(lengths), sum(n // case["hop"] + 1 for n in lengths)
    bins = case["nfft"] // 2 + 1
    fft = frames * (2.5 * case["nfft"] * math.log2(case["nfft"]) + 3 * bins)
    if kind == "dbspec":   # samples, spectrum written and read, dB written
        return {"bytes": 4 * (total + 3 * bins * frames), "flops": fft + 4 * bins * frames}
    mel = frames * (4 * bins + 4 * case["mels"])
    if kind == "chain":    # each call's input and output
        return {"bytes": 4 * (3 * total + 2 * bins * frames + 3 * case["mels"] * frames), "flops": 2 * total + fft + mel}
    if kind == "trim":     # detection reads the samples, the features those of the regions (about three fifths)
        return {"bytes": 4 * (1.6 * total + 0.6 * case["mels"] * frames), "flops": 4 * total + 0.6 * (2 * total + fft + mel)}
    read = extra if kind == "front" else 4 * total
    return {"bytes": read + 4 * case["mels"] * frames, "flops": taps + 2 * total + fft + mel}


# ---------------------------------------------------------------------- the same in 64 bits, by torch
def _mel_matrix(case):
    """[mels][bins] Slaney-scale triangles of unit area over 0 .. rate / 2."""
    bins, m, rate = case["nfft"] // 2 + 1, case["mels"], float(case["rate"])
    fsp, log_hz, step = 200.0 / 3.0, 1000.0, math.log(6.4) / 27.0
    top = log_hz / fsp + math.log(rate / 2 / log_hz) / step
    mel = np.linspace(0.0, top, m + 2)
    hz = np.where(mel >= log_hz / fsp, log_hz * np.exp(step * (mel - log_hz / fsp)), mel * fsp)
    f = np.arange(bins) * rate / case["nfft"]
    w = np.zeros((m, bins))
    for i in range(m):
        up, down = (f - hz[i]) / (hz[i + 1] - hz[i]), (hz[i + 2] - f) / (hz[i + 2] - hz[i + 1])
        w[i] = np.maximum(0.0, np.minimum(up, down)) * 2.0 / (hz[i + 2] - hz[i])
    w[:, f >= rate / 2] = 0.0
    return torch.as_tensor(w, device="cuda")


class _Exact:
    def __init__(self, case):
        n, w = case["nfft"], case["window"]
        self.case = case
        t = torch.arange(w, device="cuda", dtype=torch.float64)
        hann = 0.5 * (1.0 - torch.cos(2 * math.pi / w * (t + 0.5)))
        kt = torch.arange(w, device="cuda").unsqueeze(1) * torch.arange(n // 2 + 1, device="cuda").unsqueeze(0) % n
        angle = 2 * math.pi / n * kt.double()
        self.cos, self.sin = hann.unsqueeze(1) * torch.cos(angle), hann.unsqueeze(1) * torch.sin(angle)
        self.mel = _mel_matrix(case) if "mels" in case else None

    def spectrum(self, x):
        """[bins][frames] |X|^2 of one clip, frames centred, edges mirrored."""
        L, hop, w = len(x), self.case["hop"], self.case["window"]
        frames, out = L // hop + 1, []
        for f0 in range(0, frames, 8192):
            f = torch.arange(f0, min(f0 + 8192, frames), device="cuda")
            i = f.unsqueeze(1) * hop - w // 2 + torch.arange(w, device="cuda").unsqueeze(0)
            if L > 1:
                i = i % (2 * (L - 1))
                i = torch.where(i < L, i, 2 * (L - 1) - i)
            else:
                i = torch.zeros_like(i)
            a = x[i]
            out.append((a @ self.cos).square() + (a @ self.sin).square())
        return torch.cat(out).T

    @staticmethod
    def pre_emphasis(x, c=float(np.float32(0.97))):
        return x - c * torch.cat([x[:1], x[:-1]])

    @staticmethod
    def decibels(v, ref=1.0, multiplier=10.0, cutoff=-80.0):
        ref = float(v.max()) if ref == 0.0 else ref
        return multiplier * torch.log10(torch.clamp(v / (ref or 1.0), min=10.0 ** (cutoff / multiplier)))

    def features(self, x):
        return self.decibels(self.mel @ self.spectrum(self.pre_emphasis(x)), self.case.get("ref", 1.0))


def _resampled(x, in_rate, out_rate):
    """Windowed-sinc interpolation through the same table, positions and sums in 64 bits."""
    lut, scale, center = synth.kaiser_sinc_lut(COEFFS, LOBES)
    lut = torch.as_tensor(lut, device="cuda").double()
    n, out = _out_length(len(x), in_rate, out_rate), []
    taps = torch.arange(-LOBES, LOBES, device="cuda")
    for o0 in range(0, n, 1 << 20):
        pos = torch.arange(o0, min(o0 + (1 << 20), n), device="cuda").double() * (in_rate / out_rate)
        i = torch.ceil(pos).long().unsqueeze(1) + taps
        at = (i - pos.unsqueeze(1)) * scale + center
        k = torch.clamp(torch.floor(at).long(), 0, len(lut) - 2)
        w = lut[k] + (at - k) * (lut[k + 1] - lut[k])
        w = torch.where((i >= 0) & (i < len(x)), w, torch.zeros_like(w))
        out.append((x[torch.clamp(i, 0, len(x) - 1)] * w).sum(1))
    return torch.cat(out)


def exact(case, seed):
    kind = case["kind"]
    x, lengths = _inputs(case, seed)
    n = len(lengths)
    if kind == "trim":     # where a region begins and ends is decided in the reference's FP32 order of sums
        return None
    if kind in ("front", "resample"):
        out_rate = case["out_rate"] if kind == "resample" else OUT_16K
        longest = _out_length(int(lengths.max()), case["in_rate"], out_rate)
        mono = torch.zeros((n, _stride(int(lengths.max()))), device="cuda", dtype=torch.float64)
        res = torch.zeros((n, _stride(longest)), device="cuda", dtype=torch.float64)
        for b, l in enumerate(int(v) for v in lengths):
            mono[b, :l] = x[b, :l * case["channels"]].double().reshape(l, -1).mean(1)
            r = _resampled(mono[b, :l], case["in_rate"], out_rate)
            res[b, :len(r)] = r
        if kind == "resample":
            return mono, res
        e = _Exact(case)
        db = torch.zeros((n, case["mels"], longest // case["hop"] + 1), device="cuda", dtype=torch.float64)
        for b, l in enumerate(_out_length(int(v), case["in_rate"], out_rate) for v in lengths):
            db[b, :, :l // case["hop"] + 1] = e.features(res[b, :l])
        return db
    e, frames = _Exact(case), lengths // case["hop"] + 1
    most, bins = int(frames.max()), case["nfft"] // 2 + 1

    def zeros(rows):
        return torch.zeros((n, rows, most), device="cuda", dtype=torch.float64)

    if kind == "packed":
        return torch.cat([e.features(x[b, :int(l)].double()).reshape(-1) for b, l in enumerate(lengths)])
    if kind == "logmel":
        db = zeros(case["mels"])
        for b, l in enumerate(lengths):
            db[b, :, :frames[b]] = e.features(x[b, :int(l)].double())
        return db
    spec, db = zeros(bins), zeros(case.get("mels", bins))
    pre, mel = torch.zeros_like(x, dtype=torch.float64), zeros(case.get("mels", 0))
    for b, l in enumerate(int(v) for v in lengths):
        c = x[b, :l].double()
        f = slice(0, int(frames[b]))
        if kind == "dbspec":
            p = e.spectrum(c)
            spec[b, :, f] = p.sqrt() if case["power"] == 1 else p
            db[b, :, f] = e.decibels(spec[b, :, f], 0.0, 20.0 if case["power"] == 1 else 10.0)
            continue
        pre[b, :l] = e.pre_emphasis(c)
        spec[b, :, f] = e.spectrum(pre[b, :l])
        mel[b, :, f] = e.mel @ spec[b, :, f]
        db[b, :, f] = e.decibels(mel[b, :, f])
    return (spec, db) if kind == "dbspec" else (pre, spec, mel, db)
