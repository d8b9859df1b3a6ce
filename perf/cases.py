"""The work a program has this library do in one chunk of MelBandRoformer inference, as
single layers and blocks through the Python entry points of `mbrt`.

Sizes are those of the model the benchmark and the tests use (44.1 kHz stereo, n_fft 2048,
hop 441, 60 mel bands, 8 heads of 64, 384 features): an 8 s chunk has T = 801 frames, a
batch is 1 to 4 chunks, and shorter or longer chunks give other T.  Kinds:

  attention        fused attention over [heads, N, 64]: time (N = T) or frequency (N = 60)
  attention_qkv    the same straight from the fused qkv projection: q rotated, the output
                   gated and head-merged in the call
  attention_steps  that layer as separate calls: split + rotary, attention, gate merge
  softmax          row softmax of a stored score matrix
  stft, istft      the spectrogram in front of the model and the waveform behind it
  bands            band gather, and the complex-mask merge back onto the spectrogram
  band_split       the 60 per-band slices and their RMSNorms, and the concat of the bands
  tokens           one transformer step's elementwise work: permute, residual + RMSNorm, GELU,
                   and the mask head's GLU
  song             chunking of a whole recording: reflect pad, chunk slices, faded overlap-add
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "mbr-cuda-tile_amd"))

import mbrt  # noqa: E402

DEV = "cuda"
N_FFT, BINS, HOP = 2048, 1025, 441
HEADS, DH = 8, 64
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}
SIZE = {"f32": 4, "bf16": 2}
PRECISION = {"pair": mbrt.ATTN_P_PAIR, "bf16": mbrt.ATTN_P_BF16, "fast": mbrt.ATTN_P_BF16_FAST}


def listed():
    return [
        # time attention of an 8 s chunk, 60 bands x 8 heads, the default precision
        dict(name="attention_time", kind="attention", bh=480, n=801, p="pair", out="bf16"),
        # frequency attention of that chunk, 801 frames x 8 heads: many short sequences
        dict(name="attention_freq", kind="attention", bh=6408, n=60, p="pair", out="bf16"),
        # the time attention layer of that chunk as one call from the qkv projection
        dict(name="attention_qkv", kind="attention_qkv", b=60, n=801, p="pair", out="bf16"),
        # a 1 s chunk's layer call by call, in the single-rounded P form: latency and launches
        dict(name="attention_steps_short", kind="attention_steps", b=60, n=101, p="fast", out="bf16"),
        # stored scores of the time attention, f32: the largest call of the library
        dict(name="softmax_time", kind="softmax", rows=480 * 801, cols=801, dtype="f32"),
        # 4 stereo chunks of 8 s to spectra, and back
        dict(name="stft", kind="stft", batch=8, length=352800, hop=HOP),
        dict(name="istft", kind="istft", batch=8, length=352800, hop=HOP, dtype="f32"),
        # one stereo chunk of ragged length from the model's bf16 spectra
        dict(name="istft_stereo_bf16", kind="istft", batch=2, length=273421, hop=HOP, dtype="bf16"),
        # band split and mask merge of 4 chunks
        dict(name="bands", kind="bands", batch=4, frames=801, masks=1, dtype="f32"),
        # the per-band front end of one chunk: 60 slices, 60 norms, one concat
        dict(name="band_split", kind="band_split", batch=1, frames=801, dtype="f32"),
        # one transformer step's elementwise work on an 8 s chunk
        dict(name="tokens", kind="tokens", batch=1, frames=801, dim=384, dtype="bf16"),
        # a one-minute stereo recording of odd length in 8 s chunks, half overlapping
        dict(name="song", kind="song", channels=2, length=2645017, chunk=352800, overlap=2),
    ]


# ---- drawn cases ----------------------------------------------------------------------------

def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One case of the listed kinds: chunks of 0.5 to 16 s, batches of 1 to 4 (as far as the
    largest listed case allows), each data type and precision."""
    kind = rng.choice(["attention", "attention_qkv", "attention_steps", "softmax", "stft", "istft", "bands",
                       "band_split", "tokens", "song"])
    out = rng.choice(["bf16", "bf16", "f32"])
    dtype = rng.choice(["f32", "bf16"])
    p = rng.choice(["pair", "pair", "bf16", "fast"])
    if kind in ("attention", "attention_qkv", "attention_steps"):
        if rng.random() < 0.4:  # frequency attention: one sequence of bands per frame
            b, n = _log(rng, 50, 801), rng.choice([60, 60, rng.randint(32, 64)])
        else:                   # time attention: one sequence of frames per band
            n = _log(rng, 50, 1601)
            b = max(1, min(60, int(60 * (801 / n) ** 2)))
        if kind == "attention":
            return dict(kind=kind, bh=b * HEADS, n=n, p=p, out=out)
        return dict(kind=kind, b=b, n=n, p=p, out=out)
    if kind == "softmax":
        cols = rng.choice([60, _log(rng, 50, 1601), _log(rng, 50, 1601)])
        return dict(kind=kind, rows=_log(rng, 400, max(401, 480 * 801 * 801 // (2 * cols))), cols=cols, dtype=dtype)
    if kind == "stft":
        return dict(kind=kind, batch=rng.choice([1, 2, 2, 4, 8]), length=_log(rng, 22050, 352800),
                    hop=rng.choice([HOP, HOP, 512, 256, rng.randint(300, 1024)]))
    if kind == "istft":
        return dict(kind=kind, batch=rng.choice([1, 2, 2, 4, 8]), length=_log(rng, 22050, 352800),
                    hop=rng.choice([HOP, HOP, 512, 256, rng.randint(300, 1024)]), dtype=dtype)
    if kind == "bands":
        return dict(kind=kind, batch=rng.choice([1, 2, 4]), frames=_log(rng, 50, 801), masks=rng.choice([1, 1, 2]),
                    dtype=dtype)
    if kind == "band_split":
        batch = rng.choice([1, 1, 2])
        return dict(kind=kind, batch=batch, frames=_log(rng, 50, 801 // batch), dtype=dtype)
    if kind == "tokens":
        batch = rng.choice([1, 1, 2])
        return dict(kind=kind, batch=batch, frames=_log(rng, 50, 801 // batch), dim=rng.choice([384, 384, 256, 192]),
                    dtype=dtype)
    return dict(kind=kind, channels=rng.choice([1, 2, 2]), length=_log(rng, 400000, 2600000),
                chunk=rng.choice([352800, 352800, rng.randint(100000, 352800)]), overlap=rng.choice([2, 2, 4]))


# ---- inputs -----------------------------------------------------------------------------------

def _randn(g, shape, dtype=torch.float32, std=1.0, mean=0.0):
    return (torch.randn(shape, generator=g, device=DEV) * std + mean).to(dtype)


def _empty(shape, dtype=torch.float32):
    return torch.empty(shape, dtype=dtype, device=DEV)


def _frames(length, hop):
    return length // hop + 1


def _signal(g, batch, length):
    """Audio-like channels: a few partials and noise, peaks around 0.5."""
    t = torch.arange(length, device=DEV, dtype=torch.float64) / 44100.0
    x = torch.randn((batch, length), generator=g, device=DEV) * 0.02
    for k in range(4):
        f = 60.0 * 4.0 ** k * (1.0 + 0.1 * float(torch.rand(1, generator=g, device=DEV)))
        x += 0.1 * torch.sin(2.0 * math.pi * f * t).float() * torch.randn((batch, 1), generator=g, device=DEV)
    return x


def _spectrum(g, shape, dtype):
    """[B, F, T, 2] spectra falling with frequency, as music's do."""
    tilt = 1.0 / (1.0 + torch.arange(shape[1], device=DEV, dtype=torch.float32) / 60.0)
    return (torch.randn(shape, generator=g, device=DEV) * 8.0 * tilt[:, None, None]).to(dtype)


def _widths():
    """(freq indices, complex columns of each band) of the 60-band stereo mel layout."""
    fi, per_band = mbrt.mel_band_layout(44100.0, N_FFT, 60, 2)
    return fi, [2 * int(c) for c in per_band * (fi.size // int(per_band.sum()))]


def _band_tables():
    fi, _ = mbrt.mel_band_layout(44100.0, N_FFT, 60, 2)
    off, ind, cnt, _ = mbrt.band_csr(fi, 2 * BINS)
    return tuple(torch.from_numpy(a).to(DEV) for a in (fi, off, ind, cnt))


def _song_plan(case):
    chunk = case["chunk"]
    step = chunk // case["overlap"]
    border = chunk - step
    total = case["length"] + 2 * border
    return chunk, step, border, total, list(range(0, total, step))


def prepare(case, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    kind = case["kind"]
    st = {"case": case}
    bf16 = torch.bfloat16
    if kind == "attention":
        bh, n = case["bh"], case["n"]
        st.update(q=_randn(g, (bh, n, DH), bf16, 1.5), k=_randn(g, (bh, n, DH), bf16), v=_randn(g, (bh, n, DH), bf16),
                  y=_empty((bh, n, DH), DTYPES[case["out"]]))
    elif kind in ("attention_qkv", "attention_steps"):
        b, n = case["b"], case["n"]
        st.update(qkv=_randn(g, (b, n, 3 * HEADS * DH), bf16, 1.2), gate=_randn(g, (b, n, HEADS), bf16, 2.0),
                  y=_empty((b, n, HEADS * DH), DTYPES[case["out"]]))
        st["cos"], st["sin"] = (torch.from_numpy(t).to(DEV) for t in mbrt.rotary_tables(n, DH))
        if kind == "attention_steps":
            st.update(q=_empty((b, HEADS, n, DH), bf16), k=_empty((b, HEADS, n, DH), bf16),
                      v=_empty((b, HEADS, n, DH), bf16), o=_empty((b, HEADS, n, DH), DTYPES[case["out"]]))
    elif kind == "softmax":
        dt = DTYPES[case["dtype"]]
        st.update(x=_randn(g, (case["rows"], case["cols"]), dt, 3.0), y=_empty((case["rows"], case["cols"]), dt))
    elif kind == "stft":
        st.update(x=_signal(g, case["batch"], case["length"]), w=mbrt.hann_window(N_FFT),
                  y=_empty((case["batch"], BINS, _frames(case["length"], case["hop"]), 2)))
    elif kind == "istft":
        frames = _frames(case["length"], case["hop"])
        st.update(s=_spectrum(g, (case["batch"], BINS, frames, 2), DTYPES[case["dtype"]]), w=mbrt.hann_window(N_FFT),
                  y=_empty((case["batch"], case["length"])),
                  work=_empty(mbrt.istft_workspace_bytes(case["batch"], frames, case["hop"]) // 4))
    elif kind == "bands":
        b, t, dt = case["batch"], case["frames"], DTYPES[case["dtype"]]
        fi, off, ind, cnt = _band_tables()
        j = fi.numel()
        st.update(fi=fi, off=off, ind=ind, cnt=cnt, s=_spectrum(g, (b, 2 * BINS, t, 2), torch.float32),
                  m=[_randn(g, (b, t, 2 * j), dt, 0.5) for _ in range(case["masks"])], g=_empty((b, t, 2 * j), dt),
                  y=_empty((b * case["masks"] * 2, BINS, t, 2)))
    elif kind == "band_split":
        b, t, dt = case["batch"], case["frames"], DTYPES[case["dtype"]]
        dims = _widths()[1]
        st.update(dims=dims, x=_randn(g, (b, t, sum(dims)), dt, 4.0),
                  gamma=[_randn(g, (d,), torch.float32, 0.02, 1.0) for d in dims],
                  xb=[_empty((b, t, d), dt) for d in dims], nb=[_empty((b, t, d), dt) for d in dims],
                  y=_empty((b, t, sum(dims)), dt))
    elif kind == "tokens":
        b, t, d, dt = case["batch"], case["frames"], case["dim"], DTYPES[case["dtype"]]
        st.update(x=_randn(g, (b, t, 60, d), dt), u=_randn(g, (b, 60, t, d), dt), gamma=_randn(g, (d,), torch.float32, 0.02, 1.0),
                  h=_randn(g, (b * 60 * t, 4 * d), dt, 1.5), bias=_randn(g, (4 * d,), torch.float32, 0.1),
                  z=_randn(g, (b * t, 60 * 2 * d), dt, 1.5),
                  xp=_empty((b, 60, t, d), dt), s=_empty((b, 60, t, d), dt), n=_empty((b, 60, t, d), dt),
                  a=_empty((b * 60 * t, 4 * d), dt), glu=_empty((b * t, 60 * d), dt))
    else:  # song
        chunk, step, border, total, starts = _song_plan(case)
        c = case["channels"]
        fade = chunk // 10
        st.update(x=_signal(g, c, case["length"]).view(1, c, -1), mix=_empty((1, c, total)), piece=_empty((1, c, chunk)),
                  tails={s: _empty((1, c, total - s)) for s in starts if s + chunk > total}, wsum=_empty((total,)), acc=_empty((c, total)),
                  y=_empty((c, case["length"])),
                  # the model's output of each chunk, cut to the samples that lie in the song
                  parts=[_randn(g, (c, min(chunk, total - s)), std=0.2) for s in starts],
                  wins=[torch.from_numpy(mbrt.chunk_fade_window(chunk, fade, s == 0, s + chunk >= total)).to(DEV)[:total - s]
                        for s in starts])
    return st


# ---- one pass -------------------------------------------------------------------------------

def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "attention":
        return mbrt.attention(st["q"], st["k"], st["v"], st["y"], p_precision=PRECISION[case["p"]])
    if kind == "attention_qkv":
        b, n, _ = st["qkv"].shape
        q, k, v = st["qkv"].view(b, n, 3, HEADS, DH).unbind(2)
        return mbrt.attention_bnhd(q, k, v, st["y"], cos=st["cos"], sin=st["sin"], gate=st["gate"],
                                   p_precision=PRECISION[case["p"]])
    if kind == "attention_steps":
        b, n, _ = st["qkv"].shape
        mbrt.split_qkv_rotary(st["qkv"], st["cos"], st["sin"], st["q"], st["k"], st["v"], HEADS)
        flat = lambda t: t.view(b * HEADS, n, DH)  # noqa: E731
        mbrt.attention(flat(st["q"]), flat(st["k"]), flat(st["v"]), flat(st["o"]), p_precision=PRECISION[case["p"]])
        return mbrt.gate_merge(st["o"], st["gate"], st["y"])
    if kind == "softmax":
        return mbrt.softmax(st["x"], st["y"])
    if kind == "stft":
        return mbrt.stft(st["x"], st["w"], case["hop"], out=st["y"])
    if kind == "istft":
        return mbrt.istft(st["s"], st["w"], case["hop"], length=case["length"], out=st["y"], workspace=st["work"])
    if kind == "bands":
        mbrt.band_gather(st["s"], st["fi"], st["g"])
        mbrt.band_mask_merge(st["s"], st["m"], st["off"], st["ind"], st["cnt"], st["y"], 2)
        return st["g"], st["y"]
    if kind == "band_split":
        o = 0
        for d, xb, gamma, nb in zip(st["dims"], st["xb"], st["gamma"], st["nb"]):
            mbrt.strided_copy(st["x"][..., o:o + d], xb)
            mbrt.rms_norm(xb, gamma, nb, math.sqrt(d))
            o += d
        return mbrt.cat(st["nb"], -1, st["y"])
    if kind == "tokens":
        mbrt.strided_copy(st["x"].permute(0, 2, 1, 3), st["xp"])
        mbrt.residual_add_rms_norm(st["xp"], st["u"], st["gamma"], st["s"], st["n"], math.sqrt(case["dim"]))
        mbrt.bias_act(st["h"], st["bias"], st["a"], mbrt.ACT_GELU_STD)
        mbrt.glu(st["z"], st["glu"])
        return st["s"], st["n"], st["a"], st["glu"]
    chunk, step, border, total, starts = _song_plan(case)
    mbrt.pad(st["x"], st["mix"], [0, 0, border], reflect=True)
    mbrt.fill_(st["acc"], 0.0)
    mbrt.fill_(st["wsum"], 0.0)
    for s, part, win in zip(starts, st["parts"], st["wins"]):
        if s + chunk <= total:
            mbrt.strided_copy(st["mix"][..., s:s + chunk], st["piece"])
        else:
            mbrt.strided_copy(st["mix"][..., s:], st["tails"][s])
            mbrt.pad(st["tails"][s], st["piece"], [0, 0, 0], reflect=total - s > chunk // 2)
        # the model's forward stands here: piece -> part
        mbrt.chunk_accumulate(st["acc"], st["wsum"], part, win, s)
    mbrt.chunk_normalize(st["acc"], st["wsum"])
    mbrt.strided_copy(st["acc"][:, border:border + case["length"]], st["y"])
    return st["mix"], st["piece"], st["y"]


# ---- what a pass cannot do without --------------------------------------------------------------

def work(case):
    kind = case["kind"]
    if kind in ("attention", "attention_qkv", "attention_steps"):
        bh, n, es = case.get("bh", HEADS * case.get("b", 0)), case["n"], SIZE[case["out"]]
        nbytes = bh * n * DH * (3 * 2 + es)
        if kind != "attention":
            nbytes += bh * n * 2 + 2 * n * (DH // 2) * 4
        return {"bytes": nbytes, "flops": 4 * bh * n * n * DH}
    if kind == "softmax":
        n = case["rows"] * case["cols"]
        return {"bytes": 2 * n * SIZE[case["dtype"]], "flops": 5 * n}
    if kind in ("stft", "istft"):
        frames = _frames(case["length"], case["hop"])
        n = case["batch"] * frames
        nbytes = case["batch"] * case["length"] * 4 + N_FFT * 4 + n * BINS * 2 * SIZE[case.get("dtype", "f32")]
        return {"bytes": nbytes, "flops": int(2.5 * n * N_FFT * math.log2(N_FFT))}
    if kind == "bands":
        b, t, m, es = case["batch"], case["frames"], case["masks"], SIZE[case["dtype"]]
        cols = 2 * 3958
        spec = b * 2 * BINS * t * 8
        return {"bytes": spec + b * t * cols * es * (1 + m) + m * spec, "flops": 4 * b * t * cols * m}
    if kind == "band_split":
        n = case["batch"] * case["frames"] * 2 * 3958
        return {"bytes": 2 * n * SIZE[case["dtype"]], "flops": 4 * n}
    if kind == "tokens":
        n = case["batch"] * case["frames"] * 60 * case["dim"]
        return {"bytes": n * SIZE[case["dtype"]] * (2 + 2 + 8 + 3), "flops": n * (6 + 4 * 10 + 4)}
    chunk, step, border, total, starts = _song_plan(case)
    c = case["channels"]
    added = sum(min(chunk, total - s) for s in starts)
    return {"bytes": 4 * c * (2 * case["length"] + total + chunk + added), "flops": 2 * c * added}


# ---- tolerances and the 64-bit results -------------------------------------------------------------

def tolerance(case):
    """About four times what the start shows against 64-bit results, per data type."""
    kind = case["kind"]
    if kind in ("attention", "attention_qkv", "attention_steps"):
        if case["out"] == "bf16" or case["p"] != "pair":  # bf16 rounding of the output or of P
            return {"rel": 8e-3, "max": 6e-2}
        # P as a bf16 pair: 2^-15 of a single dominant term; where q (and k) are rotated and
        # rounded to bf16 in the call, a few of them round the other way
        return {"rel": 2e-5, "max": 2e-4} if kind == "attention" else {"rel": 1.6e-4, "max": 5e-2}
    if kind in ("softmax", "bands", "band_split", "tokens") and case["dtype"] == "bf16":
        return {"rel": 7e-3, "max": 1.6e-2}
    return {"rel": 6e-7, "max": 1.5e-5}


def _attention64(q, k, v, out):
    """q, k, v [B, N, 64] -> softmax(q k^T / 8) v in float64, a few heads at a time."""
    for i in range(0, q.shape[0], 64):
        s = torch.matmul(q[i:i + 64].double(), k[i:i + 64].double().transpose(1, 2).contiguous()) * 0.125
        out[i:i + 64] = torch.matmul(torch.softmax(s, -1), v[i:i + 64].double())
    return out


def _rms64(x, gamma, eps):
    return x * torch.rsqrt((x * x).sum(-1, keepdim=True) + eps) * gamma.double() * math.sqrt(x.shape[-1])


def exact(case, seed):
    st = prepare(case, seed)
    kind = case["kind"]
    f64 = dict(dtype=torch.float64, device=DEV)
    if kind == "attention":
        return _attention64(st["q"], st["k"], st["v"], torch.empty(st["q"].shape, **f64))
    if kind in ("attention_qkv", "attention_steps"):
        b, n, _ = st["qkv"].shape
        q, k, v = (t.permute(0, 2, 1, 3).double() for t in st["qkv"].view(b, n, 3, HEADS, DH).unbind(2))
        cos, sin = st["cos"].double(), st["sin"].double()

        def rotate(x):  # the layer's q and k are bf16
            x0, x1 = x[..., 0::2], x[..., 1::2]
            return torch.stack((x0 * cos - x1 * sin, x0 * sin + x1 * cos), -1).flatten(-2).to(torch.bfloat16)

        # the fused call takes k as the projection gives it; the steps rotate both
        q, k = rotate(q), (rotate(k) if kind == "attention_steps" else k)
        flat = lambda t: t.reshape(b * HEADS, n, DH)  # noqa: E731
        o = _attention64(flat(q), flat(k), flat(v), torch.empty((b * HEADS, n, DH), **f64))
        o = o.view(b, HEADS, n, DH).permute(0, 2, 1, 3) * torch.sigmoid(st["gate"].double())[..., None]
        return o.reshape(b, n, HEADS * DH)
    if kind == "softmax":
        return torch.softmax(st["x"].double(), -1)
    if kind == "stft":
        x = np.pad(st["x"].cpu().numpy().astype(np.float64), ((0, 0), (N_FFT // 2, N_FFT // 2)), mode="reflect")
        w = st["w"].cpu().numpy().astype(np.float64)
        out = np.empty(tuple(st["y"].shape))
        for t in range(out.shape[2]):
            z = np.fft.rfft(x[:, t * case["hop"]:t * case["hop"] + N_FFT] * w, axis=-1)
            out[:, :, t, 0], out[:, :, t, 1] = z.real, z.imag
        return out
    if kind == "istft":
        s = st["s"].double().cpu().numpy()
        w = st["w"].cpu().numpy().astype(np.float64)
        batch, _, frames, _ = s.shape
        hop, half = case["hop"], N_FFT // 2
        acc, den = np.zeros((batch, (frames - 1) * hop + N_FFT)), np.zeros((frames - 1) * hop + N_FFT)
        for t in range(frames):
            z = s[:, :, t, 0] + 1j * s[:, :, t, 1]
            acc[:, t * hop:t * hop + N_FFT] += np.fft.irfft(z, n=N_FFT, axis=-1) * w
            den[t * hop:t * hop + N_FFT] += w * w
        y = np.where(den > 1e-8, acc / np.where(den > 1e-8, den, 1.0), acc)[:, half:half + (frames - 1) * hop]
        out = np.zeros((batch, case["length"]))
        n = min(y.shape[1], out.shape[1])
        out[:, :n] = y[:, :n]
        return out
    if kind == "bands":
        fi = st["fi"].long()
        s = st["s"].double()
        b, f, t, _ = s.shape
        gathered = s[:, fi].permute(0, 2, 1, 3)
        merged = torch.zeros((b, case["masks"], f, t, 2), **f64)
        for i, m in enumerate(st["m"]):
            p = torch.view_as_complex(gathered.contiguous()) * torch.view_as_complex(m.double().view(b, t, -1, 2))
            merged[:, i].index_add_(1, fi, torch.view_as_real(p.permute(0, 2, 1).contiguous()))
        merged /= st["cnt"].double().clamp(min=1e-8)[:, None, None]
        merged = merged.view(b, case["masks"], BINS, 2, t, 2).permute(0, 1, 3, 2, 4, 5)
        return gathered.reshape(b, t, -1), merged.reshape(-1, BINS, t, 2)
    if kind == "band_split":
        return torch.cat([_rms64(x.double(), g, 1e-12) for x, g in zip(st["x"].split(st["dims"], -1), st["gamma"])], -1)
    if kind == "tokens":
        s = st["x"].permute(0, 2, 1, 3).double() + st["u"].double()
        n = _rms64(s.to(st["s"].dtype).double(), st["gamma"], 1e-12)  # normalised from the sum as stored
        h = st["h"].double() + st["bias"].double()
        a, gate = st["z"].double().chunk(2, -1)
        return s, n, 0.5 * h * (1.0 + torch.erf(h / math.sqrt(2.0))), a * torch.sigmoid(gate)
    chunk, step, border, total, starts = _song_plan(case)
    x = st["x"].double()
    mix = torch.nn.functional.pad(x, (border, border), mode="reflect")
    acc, den = torch.zeros((case["channels"], total), **f64), torch.zeros((total,), **f64)
    for s, part, win in zip(starts, st["parts"], st["wins"]):
        acc[:, s:s + part.shape[1]] += part.double() * win.double()
        den[s:s + part.shape[1]] += win.double()
    acc = torch.where(den > 1e-8, acc / den, acc)
    last = mix[..., starts[-1]:][..., :chunk]
    if last.shape[-1] == chunk:
        piece = last
    elif last.shape[-1] > chunk // 2:
        piece = torch.nn.functional.pad(last, (0, chunk - last.shape[-1]), mode="reflect")
    else:
        piece = torch.nn.functional.pad(last, (0, chunk - last.shape[-1]))
    return mix, piece, acc[:, border:border + case["length"]]
