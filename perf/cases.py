"""Performance cases of the separation framework, through its public entry points.

Model shapes are the repository's two: CONFIG_DIMS (dim 384, 62 bands, hop 441,
GELU-GLU, depth 12: the 5-minute separation benchmark) and REFERENCE_DIMS (dim
256, 90 bands, hop 512, GELU, depth 16: the reference host).  Weights are
random-init in the distribution of the synthetic packs (N(0, 0.02), gammas
N(1, 0.02)), the audio a sine mix plus noise, features N(0, 1).

Kinds of a case ("kind"):
  forward     vh_forward: one window, waveform to vocals and instrumental
  separate    vh_separate: 8 s windows every 6 s, cross-faded
  host        the native_gpu.h provider as the reference host drives it: host
              buffers, resident layers, mask estimator back in host memory
  block       vh_transformer: one axial transformer block
  band_split  vh_band_split: spectrum to band features
  mask        vh_mask_estimate: features to the complex mask
  spectral    vh_stft, then vh_istft of the masked spectrum
"""

from __future__ import annotations

import ctypes
import math
import os
import struct
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "karaoke-platform-sidecar-native_amd"))

from vocalarc_hip import native, pack  # noqa: E402
from vocalarc_hip.dims import CONFIG_DIMS, REFERENCE_DIMS  # noqa: E402

RATE = 44_100
CHUNK, STEP = 8 * RATE, 6 * RATE
DEV = "cuda:0"


def listed():
    return [
        # the shortest clip anyone separates (the reference publishes 1 s timings): launches and idle CUs count
        {"name": "forward_1s", "kind": "forward", "model": "config", "depth": 12, "samples": RATE},
        # the 5-minute benchmark's device pass: 8 windows in one pass, the last one zero-padded
        {"name": "separate_50s", "kind": "separate", "model": "config", "depth": 12, "samples": 49 * RATE + 1234,
         "batch": 8},
        # the reference host's 10 s job (T = 862) at its own shape: 16 layers and the mask estimator
        {"name": "host_10s", "kind": "host", "model": "reference", "depth": 16, "frames": 862},
        # one layer of an 8 s window: the time axis, 62 sequences of 801 frames
        {"name": "block_time_8s", "kind": "block", "model": "config", "axis": 0, "sequences": 62, "length": 801,
         "precision": "fp32"},
        # the same layer's band axis
        {"name": "block_band_8s", "kind": "block", "model": "config", "axis": 1, "sequences": 801, "length": 62,
         "precision": "fp32"},
        # the bf16 variant of the layer's time axis
        {"name": "block_time_8s_bf16", "kind": "block", "model": "config", "axis": 0, "sequences": 62, "length": 801,
         "precision": "bf16"},
        # a layer of a 1 s clip: the smallest block in use
        {"name": "block_time_1s", "kind": "block", "model": "config", "axis": 0, "sequences": 62, "length": 101,
         "precision": "fp32"},
        # the reference model's band axis: 90 bands, longer than one 64-key tile
        {"name": "block_ref_band_10s", "kind": "block", "model": "reference", "axis": 1, "sequences": 862,
         "length": 90, "precision": "fp32"},
        # the front end on 60 s in the reference's spectrum layout
        {"name": "band_split_60s", "kind": "band_split", "model": "config", "frames": 6001, "layout": 0},
        # the mask estimator of one 8 s window, frame-major
        {"name": "mask_8s", "kind": "mask", "model": "config", "frames": 801, "layout": 1},
        # the reference model's mask estimator on a 1 s clip
        {"name": "mask_ref_1s", "kind": "mask", "model": "reference", "frames": 87, "layout": 0},
        # analysis and synthesis of 60 s in the device pipeline's layout
        {"name": "spectral_60s", "kind": "spectral", "model": "config", "samples": 60 * RATE, "layout": 1},
    ]


def draw(rng):
    def between(lo, hi):  # log-uniform whole number
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    model = rng.choice(["config", "config", "reference"])
    bands = _dims(model).bands
    kind = rng.choice(["forward", "separate", "host", "block", "block", "block", "band_split", "mask", "spectral"])
    if kind == "forward":
        return {"kind": kind, "model": model, "depth": _dims(model).depth, "samples": between(RATE // 4, 8 * RATE)}
    if kind == "separate":
        return {"kind": kind, "model": "config", "depth": 12, "samples": rng.randint(9 * RATE, 48 * RATE),
                "batch": rng.randint(1, 8)}
    if kind == "host":
        return {"kind": kind, "model": "reference", "depth": 16, "frames": between(44, 1723)}
    if kind == "block":
        frames, axis = between(20, 1601), rng.randint(0, 1)
        return {"kind": kind, "model": model, "axis": axis, "sequences": frames if axis else bands,
                "length": bands if axis else frames, "precision": rng.choice(["fp32", "fp32", "bf16"])}
    if kind == "spectral":
        return {"kind": kind, "model": model, "samples": between(RATE // 4, 60 * RATE), "layout": rng.randint(0, 1)}
    return {"kind": kind, "model": model, "frames": between(20, 6001), "layout": rng.randint(0, 1)}


def _dims(model, depth=None):
    d = CONFIG_DIMS if model == "config" else REFERENCE_DIMS
    return d if depth is None else d.with_depth(depth)


def _case_dims(case):
    return _dims(case["model"], case.get("depth", 1 if case["kind"] == "block" else 0))


# ---------------------------------------------------------------- inputs

def _gen(seed, stream):
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) * 16 + stream) & 0x7FFFFFFFFFFF)
    return g


def _randn(seed, stream, *shape):
    return torch.randn(*shape, device=DEV, generator=_gen(seed, stream))


def _tensors(d, seed):
    """Every tensor of the pack in pack order, packed layout, on the device: name -> float32 [count]."""
    specs = pack.tensor_specs(d)
    values = _randn(seed, 0, sum(s.count for s in specs)).mul_(0.02)
    out, at = {}, 0
    for s in specs:
        t = values[at:at + s.count]
        out[s.name] = t.add_(1.0) if s.kind == "gamma" else t
        at += s.count
    return out


def _pack(d, seed):
    """The pack of _tensors as host bytes."""
    blob = np.empty(pack.pack_bytes(d), np.uint8)
    head = pack.header(d)
    blob[:len(head)] = np.frombuffer(head, np.uint8)
    at = len(head)
    tensors = _tensors(d, seed)
    first = next(iter(tensors.values()))
    flat = first.as_strided((sum(t.numel() for t in tensors.values()),), (1,)).cpu().numpy().view(np.uint8)
    done = 0
    for t in tensors.values():
        n = t.numel() * 4
        blob[at:at + 8] = np.frombuffer(struct.pack("<Q", t.numel()), np.uint8)
        blob[at + 8:at + 8 + n] = flat[done:done + n]
        at += 8 + n
        done += n
    return blob


def _audio(samples, seed, channels=2, partials=6):
    g = _gen(seed, 1)
    u = torch.rand(channels, partials, 3, device=DEV, generator=g, dtype=torch.float64)
    t = torch.arange(samples, device=DEV, dtype=torch.float64) / RATE
    x = 0.01 * torch.randn(channels, samples, device=DEV, generator=g, dtype=torch.float64)
    for p in range(partials):
        f, a, ph = 80 + 3920 * u[:, p, 0], 0.02 + 0.08 * u[:, p, 1], 2 * math.pi * u[:, p, 2]
        x += a[:, None] * torch.sin(2 * math.pi * f[:, None] * t[None, :] + ph[:, None])
    return x.float().contiguous()


def _spectrum_shape(d, frames, layout):
    return (d.freq_bins, d.channels, frames, 2) if layout == 0 else (d.channels, frames, d.freq_bins, 2)


class _Weights(ctypes.Structure):
    names = ("gamma", "qkv", "gate_weight", "gate_bias", "out_weight", "ff_gamma", "ff1_weight", "ff1_bias",
             "ff2_weight", "ff2_bias")
    _fields_ = [(n, ctypes.c_void_p) for n in names]


class _MaskBand(ctypes.Structure):
    _fields_ = [("first_weight", ctypes.c_void_p), ("first_bias", ctypes.c_void_p),
                ("second_weight", ctypes.c_void_p), ("second_bias", ctypes.c_void_p),
                ("input_dim", ctypes.c_int), ("first_frequency", ctypes.c_int)]


class _Host:
    """The provider with a host's pack, as the reference host holds them."""

    def __init__(self, d, blob):
        self.lib, self.blob = native.lib(), blob
        self.gpu = self.lib.native_gpu_create()
        views = pack.tensor_views(d, blob)
        ptr = lambda name: views[name].ctypes.data  # noqa: E731
        self.layers = [[_Weights(*[ptr(f"layers.{i}.{axis}.{n}") for n in _Weights.names]) for axis in range(2)]
                       for i in range(d.depth)]
        first = d.first_frequencies()
        self.masks = (_MaskBand * d.bands)(*[
            _MaskBand(ptr(f"masks.{b}.first_weight"), ptr(f"masks.{b}.first_bias"), ptr(f"masks.{b}.second_weight"),
                      ptr(f"masks.{b}.second_bias"), d.input_dims()[b], first[b]) for b in range(d.bands)])
        self.final_gamma = ptr("final_gamma")

    def __del__(self):
        if self.gpu:
            self.lib.native_gpu_destroy(self.gpu)


def prepare(case, seed):
    d, kind = _case_dims(case), case["kind"]
    s = {"kind": kind, "case": case, "d": d}
    blob = _pack(d, seed)
    if kind == "host":
        s["host"] = _Host(d, blob)
        s["data"] = _randn(seed, 2, d.bands, case["frames"], d.dim).cpu().numpy()
        s["mask"] = np.empty((d.freq_bins, d.channels, case["frames"], 2), np.float32)
        return s
    s["ctx"] = native.Context()
    s["model"] = m = native.Model(s["ctx"], d, blob)
    if case.get("precision") == "bf16":
        m.set_precision(native.PRECISION_BF16)
    if kind in ("forward", "separate", "spectral"):
        s["audio"] = _audio(case["samples"], seed)
        s["vocals"], s["instrumental"] = torch.empty_like(s["audio"]), torch.empty_like(s["audio"])
    if kind == "spectral":
        shape = _spectrum_shape(d, d.frames(case["samples"]), case["layout"])
        s["source"] = torch.empty(shape, device=DEV)
        s["mask"] = _randn(seed, 2, *shape).mul_(0.5)
    if kind == "block":
        s["x0"] = _randn(seed, 2, case["sequences"], case["length"], d.dim)
        s["x"] = torch.empty_like(s["x0"])
    if kind == "band_split":
        s["source"] = _randn(seed, 2, *_spectrum_shape(d, case["frames"], case["layout"]))
        s["out"] = torch.empty(d.bands, case["frames"], d.dim, device=DEV)
    if kind == "mask":
        s["features"] = _randn(seed, 2, case["frames"], d.bands, d.dim)
        s["mask"] = torch.empty(_spectrum_shape(d, case["frames"], case["layout"]), device=DEV)
    return s


def _run_host(s):
    h, L, T, B = s["host"], s["host"].lib, s["case"]["frames"], s["d"].bands
    ok = L.native_gpu_resident_begin(h.gpu, B, T, s["data"].ctypes.data)
    for i, (time, band) in enumerate(h.layers):
        ok &= L.native_gpu_resident_transformer(h.gpu, B, T, ctypes.addressof(time))
        ok &= L.native_gpu_resident_transpose(h.gpu, B, T)
        ok &= L.native_gpu_resident_transformer(h.gpu, T, B, ctypes.addressof(band))
        if i + 1 < len(h.layers):
            ok &= L.native_gpu_resident_transpose(h.gpu, T, B)
    ok &= L.native_gpu_resident_mask(h.gpu, T, h.final_gamma, s["mask"].ctypes.data, ctypes.addressof(h.masks), B)
    if not ok:
        raise RuntimeError("the provider declined a step")
    return s["mask"]


def run(s):
    case, kind = s["case"], s["kind"]
    if kind == "host":
        return _run_host(s)
    m = s["model"]
    if kind == "forward":
        m.forward(s["audio"], case["samples"], s["vocals"], s["instrumental"])
        return s["vocals"], s["instrumental"]
    if kind == "separate":
        m.separate(s["audio"], case["samples"], CHUNK, STEP, case["batch"], s["vocals"], s["instrumental"])
        return s["vocals"], s["instrumental"]
    if kind == "block":  # in place on a copy of the features
        s["x"].copy_(s["x0"])
        m.transformer(0, case["axis"], s["x"], case["sequences"], case["length"])
        return s["x"]
    if kind == "band_split":
        m.band_split(s["source"], case["frames"], s["out"], case["layout"])
        return s["out"]
    if kind == "mask":
        m.mask_estimate(s["features"], case["frames"], s["mask"], case["layout"])
        return s["mask"]
    m.stft(s["audio"], case["samples"], s["source"], case["layout"])
    m.istft(s["source"], s["mask"], case["samples"], s["vocals"], case["layout"])
    return s["source"], s["vocals"]


# ------------------------------------------------------------------ work

def _block_work(d, tokens, length):
    """(weight bytes, flops) of one transformer block."""
    weights = d.dim * (d.qkv_dim + d.heads + d.inner + d.ff1_out + d.ff_dim)
    return 4 * weights, 2 * tokens * weights + 4 * tokens * length * d.inner


def _mask_work(d, frames):
    weights = sum(d.mask_hidden * (d.dim + 2 * n) for n in d.input_dims())
    return 4 * weights, 2 * frames * weights


def _split_work(d, frames):
    weights = d.dim * sum(d.input_dims())
    return 4 * weights, 2 * frames * weights


def _fft_flops(d, frames):
    return 2.5 * d.n_fft * math.log2(d.n_fft) * d.channels * frames


def _windows(case):
    n = case["samples"]
    return [n] if case["kind"] == "forward" else [CHUNK] * (1 + max(0, -(-(n - CHUNK) // STEP)))


def work(case):
    d, kind = _case_dims(case), case["kind"]
    spectrum = lambda frames: 8 * d.freq_bins * d.channels * frames  # noqa: E731
    if kind in ("forward", "separate"):
        total, flops = 4 * d.channels * case["samples"] * 3, 0
        for i, n in enumerate(_windows(case)):
            T = d.frames(n)
            parts = [_split_work(d, T), _mask_work(d, T)]
            parts += [_block_work(d, T * d.bands, n_keys) for n_keys in (T, d.bands)] * d.depth
            total += sum(p[0] for p in parts) if i == 0 else 0  # weights read once
            flops += sum(p[1] for p in parts) + 2 * _fft_flops(d, T)
        return {"bytes": total, "flops": flops}
    if kind == "host":
        T = case["frames"]
        parts = [_block_work(d, T * d.bands, n) for n in (T, d.bands)] * d.depth + [_mask_work(d, T)]
        return {"bytes": 4 * T * d.bands * d.dim + spectrum(T) + sum(p[0] for p in parts),
                "flops": sum(p[1] for p in parts)}
    if kind == "block":
        tokens = case["sequences"] * case["length"]
        b, f = _block_work(d, tokens, case["length"])
        return {"bytes": b + 8 * tokens * d.dim, "flops": f}
    if kind in ("band_split", "mask"):
        T = case["frames"]
        b, f = _split_work(d, T) if kind == "band_split" else _mask_work(d, T)
        return {"bytes": b + 4 * T * d.bands * d.dim + spectrum(T), "flops": f}
    T = d.frames(case["samples"])
    return {"bytes": 3 * spectrum(T) + 8 * d.channels * case["samples"], "flops": 2 * _fft_flops(d, T)}


def tolerance(case):
    """About four times what the outputs are off exact(), measured over listed and drawn cases (a block's output is
    mostly the residual stream that entered it, so its figure is small)."""
    kind = case["kind"]
    if kind == "block":
        return {"rel": 1.2e-3} if case["precision"] == "bf16" else {"rel": 2.5e-7}
    return {"forward": {"rel": 4e-6}, "separate": {"rel": 4e-6}, "host": {"rel": 2e-6}, "band_split": {"rel": 1.1e-6},
            "mask": {"rel": 2e-6}, "spectral": {"rel": 4e-7}}[kind]


# ------------------------------------------------- the same in 64 bits

class _Exact:
    """The model's mathematics in float64 torch."""

    def __init__(self, d, seed):
        self.d, self.t = d, _tensors(d, seed)
        self.shape = {s.name: (s.out, s.inp) for s in pack.tensor_specs(d) if s.kind == "matrix"}
        n = d.n_fft
        self.window = torch.from_numpy(
            (np.float32(0.5) - np.float32(0.5) * np.cos((2 * np.pi * np.arange(n) / n).astype(np.float32)))
            .astype(np.float64)).to(DEV)

    def vec(self, name):
        return self.t[name].double()

    def mat(self, name):
        """Packed layout (32-wide output tiles [in][32], then the tail [in][tail]) -> [out][in]."""
        out, inp = self.shape[name]
        t, full = self.t[name], out // 32 * 32
        rows = [t[:full * inp].view(full // 32, inp, 32).transpose(1, 2).reshape(full, inp),
                t[full * inp:].view(inp, out - full).t()]
        return torch.cat(rows).double()

    @staticmethod
    def norm(x, gamma):
        return x * (math.sqrt(x.shape[-1]) / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-12)) * gamma

    def rope(self, x):
        """x [..., L, 64]; the angles are the reference's float32 products."""
        L, half = x.shape[-2], self.d.dim_head // 2
        freq = np.float32(1) / np.power(10000.0, np.arange(half) * 2 / self.d.dim_head).astype(np.float32)
        angle = np.arange(L, dtype=np.float32)[:, None] * freq[None, :]
        a = torch.from_numpy(angle.astype(np.float64)).to(x.device)
        c, s, e, o = torch.cos(a), torch.sin(a), x[..., 0::2], x[..., 1::2]
        return torch.stack((e * c - o * s, e * s + o * c), -1).flatten(-2)

    def block(self, layer, axis, x):
        """x [S][L][D] -> the block's output."""
        d, p = self.d, f"layers.{layer}.{axis}."
        y = self.norm(x, self.vec(p + "gamma"))
        wqkv, wg, bg = self.mat(p + "qkv"), self.mat(p + "gate_weight"), self.vec(p + "gate_bias")
        att = torch.empty(*x.shape[:2], d.inner, device=x.device, dtype=x.dtype)
        per = max(1, (1 << 28) // (d.heads * x.shape[1] * max(x.shape[1], d.inner)))
        for i in range(0, x.shape[0], per):
            q, k, v = ((y[i:i + per] @ w.t()).unflatten(-1, (d.heads, d.dim_head)).transpose(1, 2)
                       for w in wqkv.split(d.inner))
            k = self.rope(k).transpose(-1, -2).contiguous()
            o = torch.softmax(self.rope(q) @ k / math.sqrt(d.dim_head), -1) @ v.contiguous()
            g = torch.sigmoid(y[i:i + per] @ wg.t() + bg).transpose(1, 2).unsqueeze(-1)
            att[i:i + per] = (o * g).transpose(1, 2).flatten(-2)
        x = x + att @ self.mat(p + "out_weight").t()
        h = self.norm(x, self.vec(p + "ff_gamma")) @ self.mat(p + "ff1_weight").t() + self.vec(p + "ff1_bias")
        if d.ffn_glu:
            value, gate = h.chunk(2, -1)
            h = value * torch.nn.functional.gelu(gate)
        else:
            h = torch.nn.functional.gelu(h)
        return x + h @ self.mat(p + "ff2_weight").t() + self.vec(p + "ff2_bias")

    def stft(self, audio):
        """[C][n] -> complex [F][C][T] (centred, reflect-padded)."""
        d = self.d
        padded = torch.nn.functional.pad(audio.double()[None], (d.n_fft // 2, d.n_fft // 2), mode="reflect")[0]
        frames = padded.unfold(-1, d.n_fft, d.hop)
        return torch.fft.rfft(frames * self.window).permute(2, 0, 1)

    def istft(self, spec, n):
        """complex [F][C][T] -> [C][n]."""
        d, T = self.d, spec.shape[2]
        frames = torch.fft.irfft(spec.permute(1, 2, 0), n=d.n_fft) * self.window
        total = d.n_fft + d.hop * (T - 1)
        fold = lambda f: torch.nn.functional.fold(  # noqa: E731
            f.transpose(1, 2), (1, total), (1, d.n_fft), stride=(1, d.hop)).reshape(f.shape[0], total)
        env = fold((self.window * self.window).expand(1, T, d.n_fft))
        out = torch.where(env > 1e-12, fold(frames) / env.clamp_min(1e-12), 0.0)
        return out[:, d.n_fft // 2:d.n_fft // 2 + n]

    def band_split(self, spec):
        """complex [F][C][T] -> [B][T][D]."""
        out = []
        for b, (f0, w) in enumerate(zip(self.d.first_frequencies(), self.d.band_widths)):
            v = torch.view_as_real(spec[f0:f0 + w]).permute(2, 0, 1, 3).flatten(1)
            v = self.norm(v, self.vec(f"bands.{b}.gamma"))
            out.append(v @ self.mat(f"bands.{b}.weight").t() + self.vec(f"bands.{b}.bias"))
        return torch.stack(out)

    def mask(self, features):
        """final-normed [T][B][D] -> complex [F][C][T]."""
        out = []
        for b, w in enumerate(self.d.band_widths):
            h = torch.tanh(features[:, b] @ self.mat(f"masks.{b}.first_weight").t() + self.vec(f"masks.{b}.first_bias"))
            p = h @ self.mat(f"masks.{b}.second_weight").t() + self.vec(f"masks.{b}.second_bias")
            value, gate = p.chunk(2, -1)
            v = (value * torch.sigmoid(gate)).view(-1, w, self.d.channels, 2).permute(1, 2, 0, 3)
            out.append(torch.view_as_complex(v.contiguous()))
        return torch.cat(out)

    def stack(self, x):
        """[B][T][D] -> final-normed [T][B][D]."""
        for layer in range(self.d.depth):
            x = self.block(layer, 0, x).transpose(0, 1).contiguous()
            x = self.block(layer, 1, x).transpose(0, 1).contiguous()
        return self.norm(x, self.vec("final_gamma")).transpose(0, 1)

    def forward(self, audio):
        spec = self.stft(audio)
        return self.istft(spec * self.mask(self.stack(self.band_split(spec))), audio.shape[1])

    def separate(self, audio):
        n = audio.shape[1]
        count, overlap = 1 + max(0, -(-(n - CHUNK) // STEP)), CHUNK - STEP
        total, weight = (torch.zeros(c, STEP * (count - 1) + CHUNK, device=DEV, dtype=torch.float64) for c in (2, 1))
        padded = torch.nn.functional.pad(audio, (0, total.shape[1] - n))
        ramp = (torch.arange(overlap, device=DEV, dtype=torch.float64) + 0.5) / overlap
        for k in range(count):
            w = torch.ones(CHUNK, device=DEV, dtype=torch.float64)
            if k > 0:
                w[:overlap] = ramp
            if k + 1 < count:
                w[CHUNK - overlap:] = ramp.flip(0)
            at = slice(k * STEP, k * STEP + CHUNK)
            total[:, at] += w * self.forward(padded[:, at])
            weight[:, at] += w
        return (total / weight)[:, :n]


def _as_layout(spec, layout):
    """complex [F][C][T] -> real pairs in the case's layout."""
    return torch.view_as_real(spec if layout == 0 else spec.permute(1, 2, 0)).contiguous()


def _from_layout(x, layout):
    c = torch.view_as_complex(x.double().contiguous())
    return c if layout == 0 else c.permute(2, 0, 1)


def exact(case, seed):
    d, kind = _case_dims(case), case["kind"]
    e = _Exact(d, seed)
    if kind in ("forward", "separate"):
        audio = _audio(case["samples"], seed)
        vocals = e.forward(audio) if kind == "forward" else e.separate(audio)
        return vocals, audio.double() - vocals
    if kind == "host":
        x = _randn(seed, 2, d.bands, case["frames"], d.dim).double()
        return _as_layout(e.mask(e.stack(x)), 0).cpu().numpy()
    if kind == "block":
        return e.block(0, case["axis"], _randn(seed, 2, case["sequences"], case["length"], d.dim).double())
    if kind == "mask":
        features = _randn(seed, 2, case["frames"], d.bands, d.dim).double()
        return _as_layout(e.mask(features), case["layout"])
    if kind == "band_split":
        source = _randn(seed, 2, *_spectrum_shape(d, case["frames"], case["layout"]))
        return e.band_split(_from_layout(source, case["layout"]))
    audio = _audio(case["samples"], seed)
    shape = _spectrum_shape(d, d.frames(case["samples"]), case["layout"])
    spec = e.stft(audio)
    mask = _from_layout(_randn(seed, 2, *shape).mul_(0.5), case["layout"])
    return _as_layout(spec, case["layout"]), e.istft(spec * mask, case["samples"])
