"""What is timed: the calls that a program built on libstx makes, over the sizes it makes them at.

A case names one stage of a separation (its "stage") and that stage's sizes; run() is one pass of
the stage through the binding's public functions (stx.py), on buffers the program owns. exact()
restates every stage in double precision with torch alone. The sizes are the configurations of
the benchmark and the tests: HTDemucs segments (n_fft 4096, 7.8 s), RoFormer chunks (n_fft 2048,
hop 441, 352,800 samples), the MDX-Net spectra (n_fft 7680 and the smaller mixed-radix sizes),
the two models' layer ops, the song-level chunking and the resampling around a separation.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "stems.cpp_amd"))

import stx  # noqa: E402

DEV = "cuda"
F64 = torch.float64


# ------------------------------------------------------------------------------- inputs
class Rand:
    """Seeded device tensors of the values the stages meet."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(int(seed))

    def normal(self, *shape, scale=1.0):
        return torch.randn(shape, generator=self.g, device=DEV, dtype=torch.float32).mul_(scale)

    def uniform(self, *shape):
        return torch.rand(shape, generator=self.g, device=DEV, dtype=torch.float32).mul_(2.0).sub_(1.0)

    def audio(self, channels, n, rate=44100):
        """Tones below 0.4 of the rate with a noise floor, about -10 dBFS."""
        x = self.normal(channels, n, scale=0.05)
        t = torch.arange(n, device=DEV, dtype=torch.float32)
        tone = torch.rand((4, 3), generator=self.g, device=DEV).tolist()
        for f, a, p in tone:
            w = 2.0 * math.pi * (40.0 + f * 0.4 * rate) / rate
            x += (0.02 + 0.15 * a) * torch.sin(torch.remainder(t * w, 2.0 * math.pi) + 6.2831853 * p)
        return x

    def spectrum(self, *shape):
        """Complex spectra of model outputs."""
        return torch.view_as_complex(self.normal(*shape, 2, scale=0.1))


def new(*shape, dtype=torch.float32):
    return torch.empty(shape, dtype=dtype, device=DEV)


def log_int(rng, lo, hi):
    """A whole number from lo to hi, spread over its logarithm."""
    return int(min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


# ------------------------------------------------------- double-precision spectral pieces
def hann64(n):
    return torch.hann_window(n, periodic=True, dtype=F64, device=DEV)


def reflect64(x, left, right):
    return torch.nn.functional.pad(x[:, None], (left, right), mode="reflect")[:, 0]


def frames64(x, n, hop, first, count):
    """Windowed spectra [C, count, n/2+1] of the padded x, frame t at (first + t) * hop."""
    z = x[:, first * hop:].unfold(1, n, hop)[:, :count]
    return torch.fft.rfft(z * hann64(n), dim=2)


def stft64(x, n, hop):
    """torch.stft (center, reflect, not normalised), [C, T, F]."""
    return frames64(reflect64(x, n // 2, n // 2), n, hop, 0, x.shape[1] // hop + 1)


def overlap64(spec, n, hop, env_frames, frame_off):
    """Sums of the windowed inverse frames of spec [C, T, F] over the window-squared envelope of
    env_frames frames, spectrum frame t being envelope frame t + frame_off."""
    C, T, _ = spec.shape
    w = hann64(n)
    full = n + hop * (env_frames - 1)
    z = spec.clone()
    z[..., 0] = z[..., 0].real.to(z.dtype)
    z[..., -1] = z[..., -1].real.to(z.dtype)
    fr = torch.fft.irfft(z, n=n, dim=2) * w
    fold = lambda f, t: torch.nn.functional.fold(f.transpose(1, 2), (1, n + hop * (t - 1)), (1, n), stride=(1, hop))[:, 0, 0]
    y = torch.zeros((C, full), dtype=F64, device=DEV)
    y[:, frame_off * hop:frame_off * hop + n + hop * (T - 1)] = fold(fr, T)
    env = fold((w * w).expand(1, env_frames, n), env_frames)[0]
    return torch.where(env > 1e-11, y / env, torch.zeros_like(y))


def istft64(spec, n, hop):
    T = spec.shape[1]
    return overlap64(spec, n, hop, T, 0)[:, n // 2:n // 2 + hop * (T - 1)]


def demucs_spec64(x, n):
    hop = n // 4
    L = x.shape[1]
    le, pad = -(-L // hop), hop // 2 * 3
    xp = reflect64(reflect64(x, pad, pad + le * hop - L), n // 2, n // 2)
    return frames64(xp, n, hop, 2, le)[..., :-1] / math.sqrt(n)


def demucs_ispec64(spec, n, length):
    hop = n // 4
    z = torch.nn.functional.pad(torch.view_as_real(spec), (0, 0, 0, 1))
    y = overlap64(torch.view_as_complex(z), n, hop, spec.shape[1] + 4, 2) * math.sqrt(n)
    o = n // 2 + hop // 2 * 3
    return y[:, o:o + length]


def moments64(x):
    x = x.double().reshape(-1)
    return x.mean(), x.std(unbiased=True)


def fft_flops(frames, n):
    return frames * 2.5 * n * math.log2(n)


# ---------------------------------------------------------------------------- the stages
class SegmentIn:
    """One HTDemucs segment on its way into the model (the smallest call a separation makes, once
    a segment): spectrum, complex-as-channels normalise, waveform normalise."""

    N = 4096

    @staticmethod
    def draw(rng):
        return {"channels": rng.choice([1, 2]), "length": log_int(rng, 20000, 1800000)}

    @classmethod
    def prepare(cls, c, r):
        C, L = c["channels"], c["length"]
        fft = stx.FFT(cls.N)
        T, F = stx.htdemucs_frames(cls.N, L), cls.N // 2
        ws = stx.workspace(stx.lib().stx_htdemucs_norm_workspace_size(2 * C * F * T), DEV)
        return {"fft": fft, "x": r.audio(C, L), "spec": new(C, F, T, dtype=torch.complex64), "mag": new(2 * C, F, T),
                "wave": new(C, L), "stats": new(2, dtype=F64), "wstats": new(2, dtype=F64), "ws": ws}

    @staticmethod
    def run(s):
        stx.htdemucs_spec(s["fft"], s["x"], out=s["spec"])
        stx.htdemucs_cac_normalize(s["spec"], out=s["mag"], stats=s["stats"], workspace=s["ws"])
        stx.htdemucs_wave_normalize(s["x"], out=s["wave"], stats=s["wstats"], workspace=s["ws"])
        return s["mag"], s["stats"], s["wave"], s["wstats"]

    @classmethod
    def work(cls, c):
        T, F = -(-c["length"] // 1024), cls.N // 2
        return {"bytes": c["channels"] * (8 * c["length"] + 8 * F * T), "flops": fft_flops(c["channels"] * T, cls.N)}

    @classmethod
    def exact(cls, c, s):
        z = demucs_spec64(s["x"].double(), cls.N).transpose(1, 2)
        mag = torch.stack([z.real, z.imag], 1).reshape(s["mag"].shape)
        m, d = moments64(mag)
        wm, wd = moments64(s["x"])
        return ((mag - m) / (1e-5 + d), torch.stack([m, d]), (s["x"].double() - wm) / (1e-5 + wd), torch.stack([wm, wd]))

    tolerance = {"rel": 6e-7, "max": 1.6e-5}


class SegmentOut:
    """HTDemucs segments on their way out of the model, one after the other as the split loop makes
    them: denormalise, inverse spectrum of every source and channel, add the time branch."""

    N = 4096

    @staticmethod
    def draw(rng):
        return {"channels": rng.choice([1, 2, 2]), "length": log_int(rng, 40000, 600000), "sources": rng.choice([2, 4, 6]),
                "segments": rng.choice([1, 2, 3, 4])}

    @classmethod
    def prepare(cls, c, r):
        C, L, S, n = c["channels"], c["length"], c["sources"], c["segments"]
        T, F = stx.htdemucs_frames(cls.N, L), cls.N // 2
        fft = stx.FFT(cls.N)
        stats = torch.tensor([0.002, 0.7], dtype=F64, device=DEV)
        return {"fft": fft, "ox": r.normal(n, S, 2 * C, F, T), "xt": r.normal(n, S, C, L), "stats": stats,
                "spec": new(S, C, F, T, dtype=torch.complex64), "y": new(S * C, L), "out": new(n, S, C, L), "length": L}

    @staticmethod
    def run(s):
        spec = s["spec"]
        for ox, xt, out in zip(s["ox"], s["xt"], s["out"]):
            stx.htdemucs_cac_denormalize(ox, s["stats"], out=spec)
            stx.htdemucs_ispec(s["fft"], spec.view(-1, *spec.shape[2:]), s["length"], out=s["y"])
            stx.htdemucs_time_add(xt, s["y"], s["stats"], out=out)
        return s["out"]

    @classmethod
    def work(cls, c):
        T, ch = -(-c["length"] // 1024), c["channels"] * c["sources"] * c["segments"]
        return {"bytes": ch * (8 * (cls.N // 2) * T + 8 * c["length"]), "flops": fft_flops(ch * T, cls.N)}

    @classmethod
    def exact(cls, c, s):
        m, d = s["stats"].tolist()
        out = []
        for ox, xt in zip(s["ox"], s["xt"]):
            v = ox.double() * d + m
            z = torch.complex(v[:, 0::2], v[:, 1::2]).flatten(0, 1).transpose(1, 2)
            out.append(xt.double() * d + m + demucs_ispec64(z, cls.N, c["length"]).view(xt.shape))
        return torch.stack(out)

    tolerance = {"rel": 6e-7, "max": 4e-6}


def band_table(kind, n_fft, rate=44100):
    """(band sizes, bins of every band) of a RoFormer: overlapping mel triangles (Slaney scale) or
    the band-split model's consecutive runs."""
    F = n_fft // 2 + 1
    if kind == "bs":
        sizes = np.array([2] * 24 + [4] * 12 + [12] * 8 + [24] * 8 + [48] * 8 + [128, 129], dtype=np.int32)
        return sizes, np.arange(F, dtype=np.int32)
    n = int(kind[3:])
    lo, step = 1000.0 / (200.0 / 3), math.log(6.4) / 27.0
    top = lo + math.log(rate / 2.0 / 1000.0) / step
    mel = np.linspace(0.0, top, n + 2)
    hz = np.where(mel >= lo, 1000.0 * np.exp(step * (mel - lo)), mel * 200.0 / 3)
    f = np.arange(F) * (rate / n_fft)
    rows = [(f > hz[b]) & (f < hz[b + 2]) for b in range(n)]
    rows[0][0] = rows[-1][-1] = True
    return (np.array([int(m.sum()) for m in rows], dtype=np.int32),
            np.concatenate([np.nonzero(m)[0] for m in rows]).astype(np.int32))


class Roformer:
    """What both sides of a RoFormer chunk share."""

    N = 2048

    @staticmethod
    def draw(rng):
        return {"channels": rng.choice([1, 2, 2]), "length": log_int(rng, 30000, 500000), "hop": rng.choice([441, 441, 512]),
                "bands": rng.choice(["mel60", "mel60", "mel64", "bs"]), "layout": rng.choice(["t", "t", "f"]),
                "chunks": rng.choice([1, 2, 3, 4])}

    @classmethod
    def tables(cls, c):
        sizes, bins = band_table(c["bands"], cls.N)
        return stx.Bands(sizes, bins, cls.N // 2 + 1, c["channels"]), sizes, bins

    @classmethod
    def shape(cls, c):
        T, F = c["length"] // c["hop"] + 1, cls.N // 2 + 1
        return ((F, T) if c["layout"] == "f" else (T, F)), T, F

    @staticmethod
    def feat(c):
        return 2 * c["channels"] * int(band_table(c["bands"], Roformer.N)[0].sum())


class RoformerIn(Roformer):
    """RoFormer chunks on their way into the model: spectrum, band gather, every band's RMSNorm."""

    @classmethod
    def prepare(cls, c, r):
        C, L, B = c["channels"], c["length"], c["chunks"]
        bands, sizes, bins = cls.tables(c)
        tf, T, _ = cls.shape(c)
        gammas = [r.normal(2 * C * int(n)) for n in sizes]
        return {"fft": stx.FFT(cls.N), "bands": bands, "x": r.audio(B * C, L), "gammas": gammas, "hop": c["hop"], "T": T,
                "layout": stx.F_MAJOR if c["layout"] == "f" else stx.T_MAJOR,
                "spec": new(B, C, *tf, dtype=torch.complex64), "feat": new(B, bands.total_feat * T),
                "out": new(B, bands.total_feat * T)}

    @staticmethod
    def run(s):
        spec = s["spec"]
        stx.torch_stft(s["fft"], s["x"], s["hop"], layout=s["layout"], out=spec.view(-1, *spec.shape[2:]))
        s["bands"].gather(spec, s["T"], layout=s["layout"], out=s["feat"])
        s["bands"].rms_norm(s["feat"], s["T"], s["gammas"], out=s["out"])
        return spec, s["out"]

    @classmethod
    def work(cls, c):
        _, T, F = cls.shape(c)
        n = c["chunks"]
        return {"bytes": n * (4 * c["channels"] * c["length"] + 8 * c["channels"] * F * T + 4 * cls.feat(c) * T),
                "flops": fft_flops(n * c["channels"] * T, cls.N)}

    @classmethod
    def exact(cls, c, s):
        C, B = c["channels"], c["chunks"]
        z = stft64(s["x"].double(), cls.N, c["hop"])
        z = z.view(B, C, *z.shape[1:])
        sizes, bins = band_table(c["bands"], cls.N)
        parts = []
        for f, g in zip(np.split(bins, np.cumsum(sizes)[:-1]), s["gammas"]):
            v = torch.view_as_real(z[..., torch.from_numpy(f).long().to(DEV)])       # [B, C, T, size, 2]
            v = v.permute(0, 2, 3, 1, 4).reshape(B, z.shape[2], -1)
            parts.append((v / torch.sqrt(v.square().mean(2, keepdim=True) + 1e-24) * g.double()).flatten(1))
        return (z.transpose(2, 3) if c["layout"] == "f" else z), torch.cat(parts, 1)

    # The quiet bands of a frame are normalised by their own mean square: "max" is their error.
    tolerance = {"rel": 2e-6, "max": 6e-5}


class RoformerOut(Roformer):
    """RoFormer chunks on their way out of the model: the masks averaged over the bands and applied,
    then the inverse spectrum of every stem and channel."""

    @classmethod
    def draw(cls, rng):
        return dict(super().draw(rng), stems=rng.choice([1, 2, 4, 6]), zero_dc=rng.choice([True, False]))

    @classmethod
    def prepare(cls, c, r):
        C, B, S = c["channels"], c["chunks"], c["stems"]
        bands, _, _ = cls.tables(c)
        tf, T, _ = cls.shape(c)
        return {"fft": stx.FFT(cls.N), "bands": bands, "spec": r.spectrum(B, C, *tf), "masks": r.uniform(B, S, bands.total_feat * T),
                "hop": c["hop"], "T": T, "layout": stx.F_MAJOR if c["layout"] == "f" else stx.T_MAJOR, "zero_dc": c["zero_dc"],
                "est": new(B, S, C, *tf, dtype=torch.complex64), "out": new(B, S, C, c["hop"] * (T - 1))}

    @staticmethod
    def run(s):
        est, out = s["est"], s["out"]
        s["bands"].scatter_apply(s["masks"], s["spec"], s["T"], layout=s["layout"], zero_dc=s["zero_dc"], out=est)
        stx.torch_istft(s["fft"], est.view(-1, *est.shape[3:]), s["hop"], layout=s["layout"], out=out.view(-1, out.shape[3]))
        return est, out

    @classmethod
    def work(cls, c):
        _, T, F = cls.shape(c)
        ch = c["chunks"] * c["stems"] * c["channels"]
        return {"bytes": c["chunks"] * (8 * c["channels"] * F * T + 4 * c["stems"] * cls.feat(c) * T) + ch * (8 * F * T + 4 * c["length"]),
                "flops": fft_flops(ch * T, cls.N)}

    @classmethod
    def exact(cls, c, s):
        C, B, S = c["channels"], c["chunks"], c["stems"]
        _, T, F = cls.shape(c)
        sizes, bins = band_table(c["bands"], cls.N)
        z = s["spec"].to(torch.complex128)
        z = z.transpose(2, 3) if c["layout"] == "f" else z                              # [B, C, T, F]
        mask = torch.zeros((B, S, C, T, F, 2), dtype=F64, device=DEV)
        at = 0
        for f in np.split(bins, np.cumsum(sizes)[:-1]):
            n = 2 * C * len(f)
            m = s["masks"][:, :, at * T:(at + n) * T].double().view(B, S, T, len(f), C, 2).permute(0, 1, 4, 2, 3, 5)
            mask.index_add_(4, torch.from_numpy(f).long().to(DEV), m)
            at += n
        count = torch.from_numpy(np.maximum(np.bincount(bins, minlength=F), 1)).to(DEV).double()
        est = z[:, None] * (torch.view_as_complex(mask) / count)
        if c["zero_dc"]:
            est[..., 0] = 0
        # The inverse takes the spectrum as it is stored.
        y = istft64(est.to(torch.complex64).to(torch.complex128).view(B * S * C, T, F), cls.N, c["hop"])
        return (est.transpose(3, 4) if c["layout"] == "f" else est), y.view(B, S, C, -1)

    tolerance = {"rel": 8e-7, "max": 4e-6}


class DConv:
    """One HTDemucs DConv branch around its convolutions: GroupNorm + affine + GELU of the hidden
    width, GroupNorm + affine of the doubled width, GLU + LayerScale + residual. The time branch
    normalises a whole layer at once (rows 1); the frequency branch every frequency row by itself
    (rows > 1), and turns the result back to channel-major before the GLU."""

    @staticmethod
    def draw(rng):
        k = rng.randrange(4)
        C = 48 << k
        if rng.random() < 0.5:
            return {"rows": 1, "channels": C, "width": log_int(rng, 300, 400000 >> (2 * k))}
        return {"rows": 512 >> (2 * k), "channels": C, "width": rng.randint(40, 500)}

    @staticmethod
    def prepare(c, r):
        H, C, W = c["rows"], c["channels"], c["width"]
        rows = lambda n: (n, 1, W) if H == 1 else (H, n, W)
        per = lambda n: (n, 1, 1) if H == 1 else (1, n, 1)
        s = {"groups": H, "x": r.normal(C, H, W), "scale": r.normal(C, 1, 1, scale=0.1)}
        for name, n in (("h", C // 8), ("d", 2 * C)):
            a = r.normal(*rows(n))
            s[name] = (a, r.normal(*per(n)), r.normal(*per(n)), torch.empty_like(a), stx.workspace(stx.group_norm_workspace_size(a, H), DEV))
        s["turned"] = new(2 * C, H, W) if H > 1 else None
        s["out"] = new(C, H, W)
        return s

    @staticmethod
    def run(s):
        a, w, b, h, ws = s["h"]
        stx.group_norm(a, s["groups"], 1e-5, w, b, gelu=True, out=h, workspace=ws)
        a, w, b, d, ws = s["d"]
        stx.group_norm(a, s["groups"], 1e-5, w, b, out=d, workspace=ws)
        if s["turned"] is not None:
            d = stx.cont_permute(d, (0, 2, 1, 3), out=s["turned"])
        stx.glu_mul_add(s["x"], d, 2, s["scale"], out=s["out"])
        return h, s["out"]

    @staticmethod
    def work(c):
        n = c["rows"] * c["channels"] * c["width"]
        return {"bytes": n + 16 * n, "flops": 40 * n}

    @staticmethod
    def exact(c, s):
        def norm(t):
            a, w, b = (v.double() for v in t[:3])
            dims = (0, 1, 2) if c["rows"] == 1 else (1, 2)
            m = a.mean(dims, keepdim=True)
            v = (a - m).square().mean(dims, keepdim=True)
            return (a - m) / torch.sqrt(v + 1e-5) * w + b
        h, d = norm(s["h"]), norm(s["d"])
        if c["rows"] > 1:
            d = d.transpose(0, 1)
        u, v = d.chunk(2)
        return 0.5 * h * torch.special.erfc(-h / math.sqrt(2.0)), s["x"].double() + u * torch.sigmoid(v) * s["scale"].double()

    tolerance = {"rel": 1.8e-7, "max": 1.2e-6}


class Attention:
    """One RoFormer layer's ops between its matrix products, along time (N frames, B bands) or along
    the bands: RMSNorm, the q/k/v split with RoPE, softmax of the scores, the gated head merge, the
    feed-forward's bias + GELU."""

    @staticmethod
    def draw(rng):
        n, b = log_int(rng, 30, 1100), log_int(rng, 4, 801)
        return {"tokens": n, "batch": max(1, min(b, 48060 // n, 38491200 // (8 * n * n))), "heads": 8, "dh": rng.choice([32, 64, 64]), "dim": rng.choice([192, 384, 384, 512])}

    @staticmethod
    def prepare(c, r):
        N, B, H, dh, D = c["tokens"], c["batch"], c["heads"], c["dh"], c["dim"]
        return {"x": r.normal(B, N, D), "gamma": r.normal(D), "xn": new(B, N, D),
                "qkv": r.normal(B, N, 3 * H * dh), "pos": torch.arange(N, dtype=torch.int32, device=DEV), "heads": H,
                "split": (new(B, H, N, dh), new(B, H, N, dh), new(B, H, dh, N)),
                "scores": r.normal(B, H, N, N, scale=math.sqrt(dh)), "scale": 1.0 / math.sqrt(dh), "probs": new(B, H, N, N),
                "o": r.normal(B, H, N, dh), "gates": torch.sigmoid(r.normal(B, N, H, 1)), "merged": new(B, N, H, dh),
                "ff": r.normal(B, N, 4 * D), "bias": r.normal(4 * D), "act": new(B, N, 4 * D)}

    @staticmethod
    def run(s):
        stx.rms_norm(s["x"], gamma=s["gamma"], out=s["xn"])
        stx.qkv_rope_split(s["qkv"], s["pos"], s["heads"], out=s["split"])
        stx.soft_max_ext(s["scores"], scale=s["scale"], out=s["probs"])
        stx.merge_heads(s["o"], s["gates"], out=s["merged"])
        stx.gelu_erf(s["ff"], s["bias"], out=s["act"])
        return s["xn"], s["split"], s["probs"], s["merged"], s["act"]

    @staticmethod
    def work(c):
        N, B, H, dh, D = c["tokens"], c["batch"], c["heads"], c["dh"], c["dim"]
        n = B * N * (D + 3 * H * dh + H * N + H * dh + 4 * D)
        return {"bytes": 8 * n, "flops": 20 * n}

    @staticmethod
    def exact(c, s):
        N, B, H, dh = c["tokens"], c["batch"], c["heads"], c["dh"]
        x = s["x"].double()
        xn = x / torch.sqrt(x.square().mean(2, keepdim=True) + 1e-24) * s["gamma"].double()
        q, k, v = s["qkv"].double().view(B, N, 3, H, dh).permute(2, 0, 3, 1, 4)
        th = torch.arange(N, device=DEV, dtype=F64)[:, None] * 10000.0 ** (-torch.arange(0, dh, 2, device=DEV, dtype=F64) / dh)
        turn = lambda t: torch.view_as_real(torch.view_as_complex(t.reshape(B, H, N, dh // 2, 2).contiguous()) * torch.polar(torch.ones_like(th), th)).flatten(3)
        f = s["ff"].double() + s["bias"].double()
        return (xn, (turn(q), turn(k), v.transpose(2, 3)), torch.softmax(s["scores"].double() * s["scale"], 3),
                s["o"].double().transpose(1, 2) * s["gates"].double(), 0.5 * f * torch.special.erfc(-f / math.sqrt(2.0)))

    tolerance = {"rel": 1.8e-7, "max": 8e-7}


class Transformer:
    """One HTDemucs cross-transformer layer's ops between its matrix products, over the frequency or
    the time tokens: LayerNorm, softmax of the scores, bias + GELU, LayerScale + residual, the
    closing GroupNorm."""

    @staticmethod
    def draw(rng):
        return {"queries": log_int(rng, 200, 2800), "keys": log_int(rng, 200, 2800), "dim": rng.choice([384, 384, 512])}

    @staticmethod
    def prepare(c, r):
        Nq, Nk, D = c["queries"], c["keys"], c["dim"]
        x = r.normal(1, Nq, D)
        return {"x": x, "w": r.normal(D), "b": r.normal(D), "xn": new(1, Nq, D),
                "scores": r.normal(8, Nq, Nk, scale=math.sqrt(D / 8)), "scale": 1.0 / math.sqrt(D / 8), "probs": new(8, Nq, Nk),
                "ff": r.normal(Nq, 4 * D), "bias": r.normal(4 * D), "act": new(Nq, 4 * D),
                "h": r.normal(1, Nq, D), "gain": r.normal(1, 1, D, scale=0.1), "sum": new(1, Nq, D),
                "gw": r.normal(1, 1, D), "gb": r.normal(1, 1, D), "out": new(1, Nq, D),
                "ws": stx.workspace(stx.group_norm_workspace_size(x, 1), DEV)}

    @staticmethod
    def run(s):
        stx.norm(s["x"], 1e-5, s["w"], s["b"], out=s["xn"])
        stx.soft_max_ext(s["scores"], scale=s["scale"], out=s["probs"])
        stx.gelu_erf(s["ff"], s["bias"], out=s["act"])
        stx.mul_add(s["x"], s["h"], s["gain"], out=s["sum"])
        stx.group_norm(s["sum"], 1, 1e-5, s["gw"], s["gb"], out=s["out"], workspace=s["ws"])
        return s["xn"], s["probs"], s["act"], s["out"]

    @staticmethod
    def work(c):
        n = c["queries"] * (c["dim"] * 7 + 8 * c["keys"])
        return {"bytes": 8 * n, "flops": 20 * n}

    @staticmethod
    def exact(c, s):
        x = s["x"].double()
        ln = torch.nn.functional.layer_norm(x, (c["dim"],), s["w"].double(), s["b"].double(), 1e-5)
        f = s["ff"].double() + s["bias"].double()
        y = x + s["h"].double() * s["gain"].double()
        v, m = torch.var_mean(y, unbiased=False)
        return (ln, torch.softmax(s["scores"].double() * s["scale"], 2), 0.5 * f * torch.special.erfc(-f / math.sqrt(2.0)),
                (y - m) / torch.sqrt(v + 1e-5) * s["gw"].double() + s["gb"].double())

    tolerance = {"rel": 3.4e-7, "max": 2e-6}


RATES = [8000, 16000, 22050, 32000, 44100, 48000, 88200, 96000]


def resample64(x, src, dst):
    """The Kaiser-windowed sinc (beta 8.6, 32 zero crossings, 0.95 of the lower Nyquist) in double,
    from its table of 2^15 linearly interpolated points."""
    ratio = dst / src
    cutoff, steps = 0.95 * min(1.0, ratio), 1 << 15
    half = 32 / cutoff
    r = torch.clamp(torch.arange(steps + 2, device=DEV, dtype=F64) / steps, max=1.0)
    arg = math.pi * r * half * cutoff
    table = torch.where(arg < 1e-12, torch.ones_like(arg), torch.sin(arg) / torch.clamp(arg, min=1e-12)) * cutoff
    table = torch.where(r < 1, table * torch.special.i0(8.6 * torch.sqrt(1 - r * r)) / torch.special.i0(torch.tensor(8.6, device=DEV, dtype=F64)), 0.0)
    n = x.shape[1]
    out = torch.zeros((x.shape[0], int(math.floor(n * ratio + 0.5))), dtype=F64, device=DEV)
    taps = torch.arange(-int(half), int(half) + 2, device=DEV)
    for i in range(0, out.shape[1], 400000):
        k = torch.arange(i, min(i + 400000, out.shape[1]), device=DEV, dtype=F64) / ratio
        j = torch.floor(k).long()[:, None] + taps
        p = (j - k[:, None]).abs() / half * steps
        t = p.long().clamp_(max=steps)
        w = torch.where((p < steps) & (j >= 0) & (j < n), table[t] + (table[t + 1] - table[t]) * (p - t), 0.0)
        j = j.clamp_(0, n - 1)
        for c in range(x.shape[0]):
            out[c, i:i + len(k)] = (w * x[c][j]).sum(1)
    return out


class Resample:
    """A recording brought to a model's rate by itself (any pair of the usual rates, up or down)."""

    @staticmethod
    def draw(rng):
        src, dst = rng.sample(RATES, 2)
        return {"src": src, "dst": dst, "channels": rng.choice([1, 2, 2]), "length": log_int(rng, src // 4, 90 * src)}

    @staticmethod
    def prepare(c, r):
        plan = stx.Resampler(c["src"], c["dst"])
        return {"plan": plan, "x": r.audio(c["channels"], c["length"], c["src"]), "out": new(c["channels"], plan.length(c["length"]))}

    @staticmethod
    def run(s):
        return s["plan"](s["x"], out=s["out"])

    @staticmethod
    def work(c):
        out = round(c["length"] * c["dst"] / c["src"])
        taps = 2 * 32 / (0.95 * min(1.0, c["dst"] / c["src"]))
        return {"bytes": 4 * c["channels"] * (c["length"] + out), "flops": 2 * taps * out * c["channels"]}

    @staticmethod
    def exact(c, s):
        return resample64(s["x"].double(), c["src"], c["dst"])

    tolerance = {"rel": 1.2e-7, "max": 3e-7}


class Audio:
    """A whole request around a model: interleaved audio at its own rate to planar channels at the
    model's rate, the model (a gain a stem here), every stem back to the request's rate and length."""

    @staticmethod
    def draw(rng):
        return {"rate": rng.choice([22050, 32000, 48000, 48000, 96000]), "channels": rng.choice([1, 2, 2]), "stems": rng.choice([2, 4, 6]),
                "length": log_int(rng, 20000, 2000000)}

    @staticmethod
    def prepare(c, r):
        n, ch, S = c["length"], c["channels"], c["stems"]
        gains = r.normal(S)
        unit = (ctypes.c_int64 * 4)(1, 1, 1, 1), (ctypes.c_int64 * 4)(4, 4, 4, 4)

        def model(audio, channels, length, options, stems, stream):
            flat = channels * length
            ne, nb = (ctypes.c_int64 * 4)(flat, 1, 1, 1), (ctypes.c_int64 * 4)(4, 4 * flat, 4 * flat, 4 * flat)
            a = stx.Tensor(audio, ne, nb)
            for k in range(S):
                g = stx.Tensor(gains.data_ptr() + 4 * k, *unit)
                y = stx.Tensor(stems + 4 * flat * k, ne, nb)
                status = stx.lib().stx_mul(ctypes.byref(a), ctypes.byref(g), ctypes.byref(y), stream)
                if status:
                    return status
            return 0

        return {"x": r.audio(ch, n, c["rate"]).t().contiguous(), "channels": ch, "rate": c["rate"], "stems": S, "gains": gains, "model": model,
                "to": stx.Resampler(c["rate"], 44100), "from": stx.Resampler(44100, c["rate"])}

    @staticmethod
    def run(s):
        return stx.separate_audio(s["x"], s["channels"], s["rate"], stx.AUDIO_INTERLEAVED, 2, 44100, s["stems"], s["model"],
                                  to_model=s["to"], from_model=s["from"])

    @staticmethod
    def work(c):
        n, m = c["length"], round(c["length"] * 44100 / c["rate"])
        taps = 2 * 32 / (0.95 * min(1.0, 44100 / c["rate"])), 2 * 32 / (0.95 * min(1.0, c["rate"] / 44100))
        return {"bytes": 4 * n * (c["channels"] + 2 * c["stems"]), "flops": 2 * c["channels"] * m * taps[0] + 4 * c["stems"] * n * taps[1]}

    @staticmethod
    def exact(c, s):
        x = resample64(s["x"].t().double(), c["rate"], 44100)
        # The stems are the gain times the audio as it is stored.
        y = resample64(x.float().double(), 44100, c["rate"])[:, :c["length"]]
        y = torch.nn.functional.pad(y, (0, c["length"] - y.shape[1]))
        y = y.expand(2, -1) if c["channels"] == 1 else y
        return s["gains"].double()[:, None, None] * y

    tolerance = {"rel": 1.5e-7, "max": 1.2e-6}


class Song:
    """A song cut into a model's chunks and put together again: RoFormer's, MSST's and UVR's rules
    and HTDemucs' split, each with its own window."""

    @staticmethod
    def draw(rng):
        rules = rng.choice(["roformer", "msst", "uvr", "split"])
        c = {"rules": rules, "length": log_int(rng, 400000, 7938000), "stems": rng.choice([1, 2, 4])}
        if rules == "roformer":
            c.update(chunk=rng.choice([352800, 485100, 131584]), overlap=rng.choice([2, 4]))
        elif rules == "msst":
            c.update(chunk=rng.choice([261120, 130560]), overlap=rng.choice([2, 4]))
        elif rules == "uvr":
            c.update(chunk=rng.choice([261120, 130560]), overlap=0)
        else:
            c.update(chunk=343980, overlap=0)
        return c

    @staticmethod
    def prepare(c, r):
        L, S, chunk = c["length"], c["stems"], c["chunk"]
        s = {"rules": c["rules"], "mix": r.audio(2, L), "out": new(S, 2, L)}
        if c["rules"] == "split":
            s["stride"], n = stx.htdemucs_split_plan(L, chunk)
            s.update(norm=new(2, L), stats=new(2, dtype=F64), length=L, segment=chunk, ws=stx.workspace(stx.lib().stx_htdemucs_norm_workspace_size(L), DEV))
        elif c["rules"] == "uvr":
            s["plan"] = stx.UvrDemix(L, 2, chunk, 7680)
            n = s["plan"].n_chunks
        else:
            rules = stx.DEMIX_MSST if c["rules"] == "msst" else stx.DEMIX_ROFORMER
            s["plan"] = stx.Demix(L, 2, chunk, stx.demix_step(chunk, c["overlap"]), rules)
            n = s["plan"].n_chunks
        s["parts"], s["y"] = new(n, 2, chunk), r.normal(n, S, 2, chunk, scale=0.2)
        return s

    @staticmethod
    def run(s):
        if s["rules"] == "split":
            stx.htdemucs_mix_normalize(s["mix"], out=s["norm"], stats=s["stats"], workspace=s["ws"])
            stx.htdemucs_segments(s["norm"], 0, s["length"], s["segment"], s["stride"], out=s["parts"])
            y, out = s["y"], s["out"]
            stx.htdemucs_split_overlap_add(y.view(y.shape[0], -1, y.shape[3]), s["length"], s["stride"], out=out.view(-1, s["length"]))
            return s["stats"], s["parts"], out
        s["plan"].chunks(s["mix"], out=s["parts"])
        s["plan"].overlap_add(s["y"], out=s["out"])
        return s["parts"], s["out"]

    @staticmethod
    def layout(c):
        """(padded length, left border, step, [(start, length)]) of the chunks."""
        L, chunk = c["length"], c["chunk"]
        if c["rules"] == "uvr":
            gen = chunk - 7680
            total, left, step = 3840 + L + gen + 3840 - L % gen, 3840, chunk - 7680
        elif c["rules"] == "split":
            total, left, step = L, 0, int(0.75 * chunk)
        else:
            step = chunk // c["overlap"]
            border = chunk - step
            left = border if L > 2 * border and border > 0 else 0
            total = L + 2 * left
        return total, left, step, [(i, min(chunk, total - i)) for i in range(0, total, step)]

    @classmethod
    def work(cls, c):
        n = len(cls.layout(c)[3])
        return {"bytes": 8 * c["length"] + 8 * c["length"] * c["stems"] + 8 * n * c["chunk"] * (1 + c["stems"]), "flops": 6 * n * c["chunk"] * c["stems"]}

    @classmethod
    def exact(cls, c, s):
        total, left, step, table = cls.layout(c)
        L, chunk, fade = c["length"], c["chunk"], c["chunk"] // 10
        mix, y = s["mix"].double(), s["y"].double()
        n, S = y.shape[:2]
        f32 = lambda a: torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).to(DEV).double()
        i = np.arange(fade, dtype=np.float32)
        one = np.float32(1.0)
        stats = None
        if c["rules"] == "split":
            m, d = moments64(mix.mean(0).float())
            stats = torch.stack([m, d.clamp(min=1e-8)])
            mix = ((mix - m) / stats[1]).float().double()
            tri = np.minimum(np.arange(1, chunk + 1), chunk - np.arange(chunk)).astype(np.float32)
            window = f32(tri / tri.max())
        elif c["rules"] != "uvr":
            inc = one / np.float32(fade - 1)
            up = np.where(i < fade // 2, i * inc, one - (fade - 1 - i).astype(np.float32) * inc)
            down = up[::-1]
            if c["rules"] == "msst":
                down = np.where(i < fade // 2, one - inc * i, inc * (fade - 1 - i).astype(np.float32))
            ends = f32(up), f32(down)
        if c["rules"] in ("roformer", "msst") and left:
            padded = reflect64(mix, left, left)
        else:
            padded = torch.nn.functional.pad(mix, (left, total - L - left))
        parts = torch.zeros((n, 2, chunk), dtype=F64, device=DEV)
        acc = torch.zeros((S, 2, total), dtype=F64, device=DEV)
        div = torch.zeros(total, dtype=F64, device=DEV)
        for k, (a, size) in enumerate(table):
            trim = 0
            if c["rules"] == "split":
                trim = (chunk - size) // 2
                lo = a - trim
                b0, b1 = max(lo, 0), min(lo + chunk, L)
                parts[k, :, b0 - lo:b1 - lo] = mix[:, b0:b1]
                w = window[:size]
            else:
                parts[k, :, :size] = padded[:, a:a + size]
                if c["rules"] == "uvr":
                    w = 0.5 - 0.5 * torch.cos(2.0 * math.pi * torch.arange(size, device=DEV, dtype=F64) / (size - 1))
                else:
                    if size < chunk and size > chunk // 2 + (1 if c["rules"] == "roformer" else 0):
                        parts[k] = reflect64(padded[:, a:a + size], 0, chunk - size)
                    w = torch.ones(chunk, dtype=F64, device=DEV)
                    end = a + chunk >= total if c["rules"] == "roformer" else a + step >= total
                    if a > 0:
                        w[:fade] = ends[0]
                    if a == 0 or not end:
                        w[chunk - fade:] = ends[1]
                    w = w[:size]
            acc[..., a:a + size] += y[k, :, :, trim:trim + size] * w
            div[a:a + size] += w
        out = (acc / div)[..., left:left + L]
        return (parts, out) if stats is None else (stats, parts, out)

    tolerance = {"rel": 1.2e-7, "max": 3e-7}


class Spectrum:
    """A batch of signals to spectra and back at the sizes the other models take: the MDX-Net models'
    (n_fft 7680 and other products of 2, 3 and 5, a few chunks at a time) and the short frames that
    multi-band models cut whole recordings into."""

    @staticmethod
    def draw(rng):
        if rng.random() < 0.5:
            n = rng.choice([3840, 4096, 5120, 6144, 7680, 8192])
            return {"n_fft": n, "hop": rng.choice([1024, n // 4]), "channels": rng.randint(1, 12), "length": log_int(rng, 30000, 300000), "layout": rng.choice(["f", "f", "t"])}
        n = rng.choice([320, 512, 640, 960, 1024, 1536, 2048])
        return {"n_fft": n, "hop": rng.choice([n // 4, n // 2, n // 3]), "channels": rng.choice([1, 2]), "length": log_int(rng, 20000, 4000000), "layout": rng.choice(["f", "t"])}

    @staticmethod
    def prepare(c, r):
        n, hop, C = c["n_fft"], c["hop"], c["channels"]
        T, F = c["length"] // hop + 1, n // 2 + 1
        fft = stx.FFT(n, any_size=True)
        return {"fft": fft, "x": r.audio(C, c["length"]), "hop": hop, "layout": stx.F_MAJOR if c["layout"] == "f" else stx.T_MAJOR,
                "spec": new(C, *((F, T) if c["layout"] == "f" else (T, F)), dtype=torch.complex64), "out": new(C, hop * (T - 1)),
                "ws": stx.workspace(stx.istft_workspace_size(fft, C, T), DEV)}

    @staticmethod
    def run(s):
        stx.torch_stft(s["fft"], s["x"], s["hop"], layout=s["layout"], out=s["spec"])
        stx.torch_istft(s["fft"], s["spec"], s["hop"], layout=s["layout"], out=s["out"], workspace=s["ws"])
        return s["spec"], s["out"]

    @staticmethod
    def work(c):
        T, F = c["length"] // c["hop"] + 1, c["n_fft"] // 2 + 1
        return {"bytes": c["channels"] * (8 * c["length"] + 8 * F * T), "flops": 2 * fft_flops(c["channels"] * T, c["n_fft"])}

    @staticmethod
    def exact(c, s):
        z = stft64(s["x"].double(), c["n_fft"], c["hop"])
        # The inverse takes the spectrum as it is stored.
        y = istft64(z.to(torch.complex64).to(torch.complex128), c["n_fft"], c["hop"])
        return (z.transpose(1, 2) if c["layout"] == "f" else z), y

    tolerance = {"rel": 8e-7, "max": 1.6e-5}


STAGES = {"segment_in": SegmentIn, "segment_out": SegmentOut, "roformer_in": RoformerIn, "roformer_out": RoformerOut, "dconv": DConv,
          "attention": Attention, "transformer": Transformer, "resample": Resample, "audio": Audio, "song": Song, "spectrum": Spectrum}


def listed():
    return [
        # One 7.8 s HTDemucs segment, stereo: latency and launches.
        {"name": "segment_in", "stage": "segment_in", "channels": 2, "length": 343980},
        # Three segments of the four-source model.
        {"name": "segment_out", "stage": "segment_out", "channels": 2, "length": 343980, "sources": 4, "segments": 3},
        # One stereo chunk of the mel-band RoFormer.
        {"name": "roformer_in", "stage": "roformer_in", "channels": 2, "length": 352800, "hop": 441, "bands": "mel60", "layout": "t", "chunks": 1},
        # A batch of four chunks, four stems.
        {"name": "roformer_out", "stage": "roformer_out", "channels": 2, "length": 352800, "hop": 441, "bands": "mel60", "layout": "t", "chunks": 4, "stems": 4, "zero_dc": True},
        # The first encoder layer's DConv in the time and in the frequency branch (7.8 s: 336 frames).
        {"name": "dconv_time", "stage": "dconv", "rows": 1, "channels": 48, "width": 85995},
        {"name": "dconv_freq", "stage": "dconv", "rows": 512, "channels": 48, "width": 336},
        # A RoFormer time layer: 801 frames, 60 bands.
        {"name": "attention", "stage": "attention", "tokens": 801, "batch": 60, "heads": 8, "dh": 64, "dim": 384},
        # HTDemucs' frequency tokens, attending to themselves.
        {"name": "transformer", "stage": "transformer", "queries": 2688, "keys": 2688, "dim": 384},
        # Half a minute of 48 kHz stereo through a four-stem model at 44.1 kHz.
        {"name": "audio", "stage": "audio", "rate": 48000, "channels": 2, "stems": 4, "length": 1440003},
        # A three-minute song, four stems, overlap 4.
        {"name": "song", "stage": "song", "rules": "roformer", "length": 7938000, "stems": 4, "chunk": 352800, "overlap": 4},
        # Four stereo MDX-Net chunks, and a minute of stereo in short frames.
        {"name": "spectrum_mdx", "stage": "spectrum", "n_fft": 7680, "hop": 1024, "channels": 8, "length": 261120, "layout": "f"},
        {"name": "spectrum_short", "stage": "spectrum", "n_fft": 960, "hop": 480, "channels": 2, "length": 2646001, "layout": "f"},
    ]


def draw(rng):
    stage = rng.choice(sorted(STAGES))
    return dict(STAGES[stage].draw(rng), stage=stage)


def prepare(case, seed):
    return case["stage"], STAGES[case["stage"]].prepare(case, Rand(seed))


def run(state):
    return STAGES[state[0]].run(state[1])


def work(case):
    return STAGES[case["stage"]].work(case)


def tolerance(case):
    """About four times the error against exact() that the stages showed over the listed cases and
    24 drawn ones (single-precision sums and roundings)."""
    return dict(STAGES[case["stage"]].tolerance)


def exact(case, seed):
    stage = STAGES[case["stage"]]
    return stage.exact(case, stage.prepare(case, Rand(seed)))
