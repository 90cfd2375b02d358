"""Performance cases of the FastConformer framework, run through its public Python binding (pkx).

A case is one call (or one chain of calls) of a speech-recognition program:

  mel      log-mel front end: PCM clips on the device -> normalised features
  sub      dw-striding subsampling x8: features -> encoder frames
  layer    one conformer block on a residual stream
  attn     one relative-position attention (q/k/v, positional, out projections)
  enc      a whole offline encoder and the CTC head: features -> log-probabilities
  stream   one step of the cache-aware streaming encoder for S streams
  greedy   batched greedy TDT decode of encoder frames

Weights are seeded random ones of the architecture, loaded once per model and
kept, as a program keeps its checkpoint; every input depends on the seed.
exact() restates each path in torch float64 on the stored (dequantised) weights.
"""
import functools
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PY = os.path.join(ROOT, "parakeet.cpp_amd", "python")
if _PY not in sys.path:
    sys.path.insert(0, _PY)

import pk_model as pm  # noqa: E402
import pkx  # noqa: E402

# The framework's own shapes: the 0.6B and 110M offline encoders of its
# benchmark, and the cache-aware streaming model.
SHAPES = {
    "0.6b": dict(d_model=1024, n_heads=8, ff_dim=4096, conv_kernel=9, n_mels=128, sub_channels=256, vocab_size=1024,
                 attn_bias=False, ff_bias=False, conv_bias=False, n_layers=24),
    "110m": dict(d_model=512, n_heads=8, ff_dim=2048, conv_kernel=9, n_mels=80, sub_channels=256, vocab_size=1024,
                 n_layers=17),
}
STREAM_WARM = 40      # windows before the measured step: the 70-frame attention cache is full
SAMPLE_RATE, HOP = 16000, 160


def listed():
    return [
        # a batch of 10 s clips from a file queue, 128 features
        {"name": "mel_b16_10s", "kind": "mel", "B": 16, "samples": 160000, "n_mels": 128, "ragged": False},
        # one short voice command for the 80-feature model: the smallest call
        {"name": "mel_b1_3s", "kind": "mel", "B": 1, "samples": 51234, "n_mels": 80, "ragged": False},
        # the encoder's input stage on a ragged batch of clips up to 10 s
        {"name": "sub_q8_b16_ragged", "kind": "sub", "shape": "0.6b", "weights": "q8_0", "B": 16, "T": 1001, "ragged": True},
        # one utterance of 10 s through a block: interactive transcription
        {"name": "layer_q8_b1_10s", "kind": "layer", "shape": "0.6b", "weights": "q8_0", "B": 1, "T": 125, "ragged": False},
        # the benchmark's batch through a block with q4_K weights, ragged lengths
        {"name": "layer_q4k_b16_ragged", "kind": "layer", "shape": "0.6b", "weights": "q4_k", "B": 16, "T": 227, "ragged": True},
        # long recordings (5 minutes each): the quadratic attention
        {"name": "layer_q8_b4_300s", "kind": "layer", "shape": "0.6b", "weights": "q8_0", "B": 4, "T": 3750, "ragged": False},
        # attention of 30 s clips, f16 weights
        {"name": "attn_f16_b8_30s", "kind": "attn", "shape": "0.6b", "weights": "f16", "B": 8, "T": 375, "ragged": False},
        # the benchmark: the whole 0.6B encoder, q8_0, 16 x 10 s, and its CTC head
        {"name": "enc_0.6b_q8_b16_10s", "kind": "enc", "shape": "0.6b", "weights": "q8_0", "B": 16, "T": 1000, "ragged": False},
        # the exact-precision path on one utterance: the whole 110M encoder in f32
        {"name": "enc_110m_f32_b1_10s", "kind": "enc", "shape": "110m", "weights": "f32", "B": 1, "T": 1000, "ragged": False},
        # a microphone: one stream, 160 ms of new audio per step
        {"name": "stream_q8_s1", "kind": "stream", "weights": "q8_0", "S": 1},
        # a streaming server at its benchmark's load
        {"name": "stream_q8_s256", "kind": "stream", "weights": "q8_0", "S": 256},
        # greedy TDT decode of the benchmark's encoder output
        {"name": "greedy_tdt_b16_10s", "kind": "greedy", "B": 16, "T": 125, "ragged": True},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["mel", "sub", "layer", "attn", "enc", "stream", "greedy"])
    ragged = rng.random() < 0.5
    if kind == "mel":
        return {"kind": kind, "B": _log_int(rng, 1, 32), "samples": _log_int(rng, 8000, 480000),
                "n_mels": rng.choice([80, 128]), "ragged": ragged}
    if kind == "stream":
        return {"kind": kind, "weights": rng.choice(["q8_0", "f16"]), "S": _log_int(rng, 1, 256)}
    if kind == "greedy":
        return {"kind": kind, "B": _log_int(rng, 1, 32), "T": _log_int(rng, 12, 375), "ragged": ragged}
    shape, weights = rng.choice([("0.6b", "q8_0"), ("0.6b", "q4_k"), ("0.6b", "f16"), ("110m", "q8_0"), ("110m", "f32")])
    if kind == "enc":
        shape, weights = rng.choice([("0.6b", "q8_0"), ("110m", "f16"), ("110m", "f32")])
    # frames after subsampling: 1 s to 30 s for the encoder's calls, to 5 minutes for a block
    T = _log_int(rng, 12, 375 if kind in ("enc", "sub") or weights == "f32" else 3750)
    B = min(_log_int(rng, 1, 16), max(1, (2000 if weights == "f32" or kind == "enc" else 8000) // T))
    if kind in ("enc", "sub"):
        T = 8 * T - rng.randrange(8)
    return {"kind": kind, "shape": shape, "weights": weights, "B": B, "T": T, "ragged": ragged}


# ---------------------------------------------------------------------------
# models and inputs
# ---------------------------------------------------------------------------
def _model_key(case):
    k = case["kind"]
    if k == "stream":
        return ("eou", case["weights"], 17, False)
    if k == "greedy":
        return ("0.6b", "q8_0", 1, "decoder")
    return (case["shape"], case["weights"], SHAPES[case["shape"]]["n_layers"] if k == "enc" else 1, k == "enc")


@functools.lru_cache(maxsize=4)
def _host_model(key):
    shape, weights, layers, heads = key
    if shape == "eou":
        return pm.synthesize(pm.eou_config(), weights, heads=False, bn_random=True)
    m = pm.synthesize(pm.Config(**dict(SHAPES[shape], n_layers=layers)), weights, heads=bool(heads), bn_random=True)
    if heads == "decoder":
        pm.add_prediction(m)
    return m


@functools.lru_cache(maxsize=None)
def _device_model(key):
    return pkx.Model.from_tensors(_host_model(key), pkx.PREC_AUTO)


@functools.lru_cache(maxsize=None)
def _front_end(n_mels):
    c = pm.Config(n_mels=n_mels)
    return pkx.Mel.create(c.n_fft, c.win_length, c.hop_length, n_mels, pm.hann_window(c.win_length),
                          pm.mel_filterbank(c.sample_rate, c.n_fft, n_mels))


@functools.lru_cache(maxsize=None)
def _stream():
    return pkx.Stream()


class _Dev:
    """A torch tensor as the binding's device array (address, shape, dtype)."""

    def __init__(self, t):
        self.t, self.ptr, self.shape = t, t.data_ptr(), tuple(t.shape)
        self.dtype = np.dtype(str(t.dtype).replace("torch.", ""))


def _gen(seed, salt):
    return torch.Generator(device="cuda").manual_seed((int(seed) * 1000003 + salt) % (1 << 62))


def _randn(seed, salt, *shape):
    return torch.randn(shape, generator=_gen(seed, salt), device="cuda", dtype=torch.float32)


def _lengths(case, seed, full):
    """Lengths of a batch: all full, or spread evenly down to a fifth, in the seed's order."""
    B = case["B"]
    if not case["ragged"]:
        return np.full(B, full, np.int32)
    v = np.array([max(2, full - (full * 4 * i) // (5 * B)) for i in range(B)], np.int32)
    return np.random.default_rng(seed).permutation(v).astype(np.int32)


def _pcm(case, seed):
    """Noise under a syllable-rate envelope, quiet stretches among it: [B][samples]."""
    B, n = case["B"], case["samples"]
    x = _randn(seed, 1, B, n)
    knots = torch.rand((B, n // 2000 + 2), generator=_gen(seed, 2), device="cuda")
    env = torch.nn.functional.interpolate((knots ** 3)[:, None], size=n, mode="linear", align_corners=True)[:, 0]
    x = 0.2 * x * env
    lens = _lengths(case, seed, n)
    for b in range(B):
        x[b, int(lens[b]):] = 0
    return x.contiguous(), lens


def _features(case, seed, n_mels):
    lens = _lengths(case, seed, case["T"])
    x = _randn(seed, 3, case["B"], n_mels, case["T"])
    for b in range(case["B"]):
        x[b, :, int(lens[b]):] = 0
    return x, lens


def _windows(case, seed, n_mels):
    """The audio of the streams: the first window's 9 frames, then 16 new ones per step."""
    return _randn(seed, 4, case["S"], n_mels, 16 * (STREAM_WARM - 1) + 25)


def prepare(case, seed):
    k, f32 = case["kind"], torch.float32
    st = {"case": case, "stream": _stream()}
    if k == "mel":
        pcm, lens = _pcm(case, seed)
        mel = _front_end(case["n_mels"])
        T = mel.frames(case["samples"])
        st.update(mel=mel, pcm=_Dev(pcm), lens=lens, T=T,
                  out=_Dev(torch.empty((case["B"], case["n_mels"], T), device="cuda", dtype=f32)))
        torch.cuda.synchronize()
        return st
    m = _device_model(_model_key(case))
    D = m.cfg.d_model
    st["model"] = m
    if k in ("sub", "enc"):
        x, st["lens"] = _features(case, seed, m.cfg.n_mels)
        Tp = pkx.subsampled_len(case["T"])
        st.update(x=_Dev(x), out=_Dev(torch.empty((case["B"], Tp, D), device="cuda", dtype=f32)))
        if k == "enc":
            M, V = case["B"] * Tp, m.cfg.vocab_size + 1
            st.update(M=M, logp=_Dev(torch.empty((case["B"], Tp, V), device="cuda", dtype=f32)),
                      best=_Dev(torch.empty((case["B"], Tp), device="cuda", dtype=torch.int32)))
    elif k in ("layer", "attn"):
        B, T = case["B"], case["T"]
        st.update(x=_Dev(_randn(seed, 5, B, T, D)), lens=_lengths(case, seed, T), pe=_Dev(_pos_table(T, D).float()),
                  out=_Dev(torch.empty((B, T, D), device="cuda", dtype=f32)))
    elif k == "greedy":
        lens = _lengths(case, seed, case["T"])
        st.update(x=_Dev(_randn(seed, 6, case["B"], case["T"], D)), lens=lens, durations=(0, 1, 2, 3, 4))
    else:
        S = case["S"]
        audio = _windows(case, seed, m.cfg.n_mels)
        torch.cuda.synchronize()
        enc = pkx.Streaming(m, n_streams=S, max_window=25, stream=st["stream"])
        out = _Dev(torch.empty((S, enc.chunk_len(9), D), device="cuda", dtype=f32))
        for i in range(STREAM_WARM):
            lo, hi = (0, 9) if i == 0 else (16 * (i - 1), 16 * (i - 1) + 25)
            w = _Dev(audio[:, :, lo:hi].contiguous())
            if enc.chunk_len(hi - lo) != out.shape[1]:
                out = _Dev(torch.empty((S, enc.chunk_len(hi - lo), D), device="cuda", dtype=f32))
            torch.cuda.synchronize()
            enc.step(w, out, stream=st["stream"])
            torch.cuda.synchronize()
        st.update(enc=enc, out=out, x=_Dev(audio[:, :, 16 * (STREAM_WARM - 1):].contiguous()))
    torch.cuda.synchronize()
    return st


def run(st):
    case, s = st["case"], st["stream"]
    k = case["kind"]
    if k == "mel":
        st["mel"].forward(st["pcm"], st["lens"], st["out"], st["T"], stream=s)
        return st["out"].t
    if k == "stream":
        st["enc"].step(st["x"], st["out"], stream=s)
        return st["out"].t
    m = st["model"]
    if k == "sub":
        m.subsampling_forward(st["x"], st["lens"], st["out"], stream=s)
    elif k == "layer":
        m.conformer_layer(0, st["x"], st["lens"], st["out"], stream=s, pos_emb=st["pe"])
    elif k == "attn":
        m.relpos_attention(0, st["x"], st["lens"], st["out"], stream=s, pos_emb=st["pe"])
    elif k == "enc":
        m.encoder_forward(st["x"], st["lens"], st["out"], stream=s)
        m.ctc(st["out"], st["M"], st["logp"], st["best"], stream=s)
        return [st["out"].t, st["logp"].t]
    else:
        items = m.transducer_greedy(st["x"], st["lens"], durations=st["durations"], stream=s)
        # one rectangle per field for the batch, as a program hands them on: ids, frames, confidences, spans
        got = [np.full((case["B"], 10 * case["T"]), pad, dt) for pad, dt in ((-1, np.int32), (-1, np.int32),
                                                                              (0, np.float32), (-1, np.int32))]
        for b, item in enumerate(items):
            for rect, v in zip(got, item):
                rect[b, :len(v)] = v
        return got
    return st["out"].t


# ---------------------------------------------------------------------------
# work and tolerance
# ---------------------------------------------------------------------------
_BYTES = {"f32": 4.0, "f16": 2.0, "q8_0": 34 / 32, "q4_k": 144 / 256}


def _layer_work(c, wb, M, B, T, attn_only=False):
    D, FF = c.d_model, c.ff_dim
    fl = 2.0 * M * D * D * 4 + 2.0 * (2 * T - 1) * D * D + 6.0 * B * T * T * D
    by = 5.0 * D * D * wb
    if not attn_only:
        fl += 4 * 2.0 * M * D * FF + 2.0 * M * D * 3 * D + 2.0 * M * D * c.conv_kernel
        by += 4.0 * D * FF * wb + 3.0 * D * D * (4 if wb == 4 else 2)
    return fl, by


def _sub_work(c, wb, B, T, causal=False):
    h = lambda t: t // 2 + 1 if causal else (t - 1) // 2 + 1  # noqa: E731
    T1, T2, T3 = h(T), h(h(T)), h(h(h(T)))
    F1, F2, F3 = h(c.n_mels), h(h(c.n_mels)), h(h(h(c.n_mels)))
    C = c.sub_channels
    fl = 2.0 * B * (T1 * F1 * C * 9 + T2 * F2 * C * (9 + C) + T3 * F3 * C * (9 + C) + T3 * C * F3 * c.d_model)
    return fl, C * F3 * c.d_model * wb + 2.0 * C * C * 4, T3


def work(case):
    k = case["kind"]
    if k == "mel":
        B, n, F = case["B"], case["samples"], case["n_mels"]
        T = 1 + n // HOP
        # a 512-point real FFT and the filterbank's ~514 nonzeros per frame
        return {"bytes": 4.0 * B * (n + F * T), "flops": B * T * (2.5 * 512 * 9 + 2 * 514 + 3 * 257 + 400 * 3)}
    if k == "stream":
        c, S, wb = pm.eou_config(), case["S"], _BYTES[case["weights"]]
        D, L, M = c.d_model, c.n_layers, 2 * S
        fl, by, _ = _sub_work(c, wb, S, 25, True)
        fl += L * (2.0 * M * D * (4 * c.ff_dim + 7 * D) + 6.0 * S * 2 * 72 * D)
        by += L * (4.0 * D * c.ff_dim * wb + 4.0 * D * D * wb + 3.0 * D * D * 2)
        # per stream: f16 key / value rings read, two rows written, f32 conv history read and rewritten
        by += S * L * (2.0 * 70 * D * 2 + 2 * 2 * D * 2 + 2 * 8 * D * 4) + S * (25 * c.n_mels * 4 + 2 * D * 4)
        return {"bytes": by, "flops": fl}
    if k == "greedy":
        B, T, H, D = case["B"], case["T"], 640, 1024
        w = 2 * 4 * H * 2 * H + H * H + 1030 * H
        # about 0.95 decode steps per frame with these weights
        return {"bytes": 4.0 * (w + D * H + B * T * D), "flops": 2.0 * B * T * D * H + 2.0 * w * B * 0.95 * T}
    c = _config(case)
    B, wb = case["B"], _BYTES[case["weights"]]
    if k in ("layer", "attn"):
        T = case["T"]
        fl, by = _layer_work(c, wb, B * T, B, T, k == "attn")
        return {"bytes": by + 4.0 * c.d_model * (2 * B * T + 2 * T - 1), "flops": fl}
    fl, by, T3 = _sub_work(c, wb, B, case["T"])
    by += 4.0 * B * (case["T"] * c.n_mels + T3 * c.d_model)
    if k == "enc":
        lf, lb = _layer_work(c, wb, B * T3, B, T3)
        V = c.vocab_size + 1
        fl += c.n_layers * lf + 2.0 * B * T3 * c.d_model * V
        by += c.n_layers * lb + 4.0 * (V * c.d_model + B * T3 * V)
    return {"bytes": by, "flops": fl}


def _config(case):
    return pm.Config(**dict(SHAPES[case["shape"]], n_layers=_model_key(case)[2]))


def tolerance(case):
    """About four times the float32 / float16 paths' measured distance from exact()."""
    k = case["kind"]
    if k == "mel":       # f64 arithmetic, f32 roundings: 2e-7
        return {"rel": 2e-6, "max": 1e-4}
    if k == "greedy":    # confidences in f32 sums; the decisions are the same
        return {"rel": 1e-5, "max": 4e-4, "differ": 0.0}
    if k == "stream":    # 17 blocks on f16 operands: 5.6e-4
        return {"rel": 2.5e-3}
    if case["weights"] == "f32":     # 17 blocks of f32 sums: 8e-7
        return {"rel": 5e-6}
    # f16 operands: subsampling 1.9e-4, a block 2.7e-4, attention alone 5.7e-4, 24 blocks 9.5e-4
    return {"rel": {"sub": 8e-4, "layer": 1.1e-3, "attn": 2.3e-3, "enc": 4e-3}[k]}


# ---------------------------------------------------------------------------
# float64 restatement
# ---------------------------------------------------------------------------
F64 = torch.float64


def _dequant(t):
    """A stored tensor's values in float64 on the GPU, torch shape."""
    if t.gtype == pm.GGML_F32:
        return torch.from_numpy(np.array(t.data, np.float32)).cuda().double().reshape(t.shape)
    raw = torch.from_numpy(np.ascontiguousarray(t.data)).cuda() if t.gtype != pm.GGML_F16 else None
    if t.gtype == pm.GGML_F16:
        return torch.from_numpy(np.ascontiguousarray(t.data).view(np.float16)).cuda().double().reshape(t.shape)
    if t.gtype == pm.GGML_Q8_0:
        b = raw.reshape(-1, 34)
        d = b[:, :2].contiguous().view(torch.float16).double()
        return (d * b[:, 2:].contiguous().view(torch.int8).double()).reshape(t.shape)
    b = raw.reshape(-1, 144)
    d = b[:, :2].contiguous().view(torch.float16).double()
    dmin = b[:, 2:4].contiguous().view(torch.float16).double()
    s = b[:, 4:16].int()
    lo, mid, hi = s[:, 0:4], s[:, 4:8], s[:, 8:12]
    sc = torch.cat([lo & 63, (hi & 15) | ((lo >> 6) << 4)], 1).double()
    mn = torch.cat([mid & 63, (hi >> 4) | ((mid >> 6) << 4)], 1).double()
    q = b[:, 16:].int().reshape(-1, 4, 32)
    q = torch.stack([q & 15, q >> 4], 2).reshape(-1, 8, 32).double()
    return ((d * sc)[:, :, None] * q - (dmin * mn)[:, :, None]).reshape(t.shape)


class _Exact:
    """The encoder's arithmetic in float64 (batched masks; causal for the streaming model)."""

    def __init__(self, key):
        self.m = _host_model(key)
        self.c = self.m.cfg
        self.causal = bool(self.c.causal_downsampling)

    def g(self, name):
        t = self.m.tensors.get(name)
        return None if t is None else _dequant(t)

    def lin(self, x, w, b=None):
        W = self.g(w)
        y = x @ W.reshape(W.shape[0], -1).t()
        bias = self.g(b) if b else None
        return y if bias is None else y + bias

    def ln(self, x, name):
        mu = x.mean(-1, keepdim=True)
        v = ((x - mu) ** 2).mean(-1, keepdim=True)
        return (x - mu) / torch.sqrt(v + 1e-5) * self.g(name + ".weight") + self.g(name + ".bias")

    def sub(self, mel, lens):
        """mel [B][F][T]; lens: entry valid frames.  -> [B][T'][D], valid per item."""
        p = "encoder.pre_encode."
        lo = 2 if self.causal else 1
        half = (lambda v: v // 2 + 1) if self.causal else (lambda v: (v - 1) // 2 + 1)
        x = mel.double().transpose(1, 2)[:, None]
        v = np.asarray(lens, np.int64)

        def mask(x, v):
            t = torch.arange(x.shape[2], device=x.device)[None, :] < torch.as_tensor(v, device=x.device)[:, None]
            return x * t[:, None, :, None]

        def conv(x, w, b):       # 3x3, stride 2, per channel (one input channel: broadcast)
            x = torch.nn.functional.pad(x, (lo, 1, lo, 1))
            ho, wo = (x.shape[2] - 3) // 2 + 1, (x.shape[3] - 3) // 2 + 1
            W = self.g(p + w)
            y = self.g(p + b)[None, :, None, None]
            for i in range(3):
                for j in range(3):
                    y = y + W[None, :, 0, i, j, None, None] * x[:, :, i:i + 2 * ho - 1:2, j:j + 2 * wo - 1:2]
            return y

        def pw(x, w, b):
            W = self.g(p + w)[:, :, 0, 0]
            y = torch.matmul(W, x.reshape(x.shape[0], x.shape[1], -1)).reshape(x.shape)
            return torch.relu(y + self.g(p + b)[None, :, None, None])

        x = torch.relu(conv(mask(x, v), "conv.0.weight", "conv.0.bias"))
        v = half(v)
        x = pw(conv(mask(x, v), "conv.2.weight", "conv.2.bias"), "conv.3.weight", "conv.3.bias")
        v = half(v)
        x = pw(conv(mask(x, v), "conv.5.weight", "conv.5.bias"), "conv.6.weight", "conv.6.bias")
        v = half(v)
        x = mask(x, v)
        x = x.transpose(1, 2).reshape(x.shape[0], x.shape[2], -1)
        return self.lin(x, p + "out.weight", p + "out.bias"), np.minimum(v, x.shape[1])

    def attention(self, i, x, pe, valid):
        c, p = self.c, "encoder.layers.%d.self_attn." % i
        B, T, D = x.shape
        H, dk = c.n_heads, D // c.n_heads
        q, k, v = (self.lin(x, p + "linear_%s.weight" % n, p + "linear_%s.bias" % n).reshape(B, T, H, dk).permute(0, 2, 1, 3).contiguous()
                   for n in "qkv")
        pp = self.lin(pe, p + "linear_pos.weight").reshape(-1, H, dk).permute(1, 2, 0).contiguous()     # [H][dk][2T-1]
        u, w = (self.g(p + "pos_bias_" + n).reshape(H, 1, dk) for n in "uv")
        j = torch.arange(T, device=x.device)
        ctx = torch.zeros((B, T, D), dtype=F64, device=x.device)
        for b in range(B):
            kt = k[b].transpose(1, 2).contiguous()
            for lo in range(0, int(valid[b]), 1024):
                r = torch.arange(lo, min(lo + 1024, int(valid[b])), device=x.device)
                bd = torch.matmul(q[b][:, r] + w, pp)
                at = (T - 1 - r[:, None] + j[None, :]).expand(H, -1, -1)
                s = (torch.matmul(q[b][:, r] + u, kt) + torch.gather(bd, 2, at)) / math.sqrt(dk)
                off = (j >= int(valid[b]))[None, :].expand(len(r), -1)
                if self.causal:      # chunked-limited window
                    n = c.att_context_right + 1
                    d = r[:, None] // n - j[None, :] // n
                    off = off | (d < 0) | (d > c.att_context_left // n)
                a = torch.softmax(s.masked_fill(off, float("-inf")), -1)
                ctx[b, r] = torch.matmul(a, v[b]).permute(1, 0, 2).reshape(len(r), D)
        return self.lin(ctx, p + "linear_out.weight", p + "linear_out.bias")

    def conv(self, i, x, valid):
        c, p = self.c, "encoder.layers.%d.conv." % i
        B, T, D = x.shape
        y = self.lin(x, p + "pointwise_conv1.weight", p + "pointwise_conv1.bias")
        y = y[..., :D] * torch.sigmoid(y[..., D:])
        y = y * (torch.arange(T, device=x.device)[None, :] < torch.as_tensor(valid, device=x.device)[:, None])[..., None]
        K = c.conv_kernel
        y = torch.nn.functional.pad(y, (0, 0, K - 1, 0) if self.causal else (0, 0, K // 2, K // 2))
        W = self.g(p + "depthwise_conv.weight")[:, 0]
        z = sum(W[:, t] * y[:, t:t + T] for t in range(K))
        b = self.g(p + "depthwise_conv.bias")
        z = z if b is None else z + b
        if c.conv_norm_type == "layer_norm":
            z = self.ln(z, p + "batch_norm")
        else:
            z = (z - self.g(p + "batch_norm.running_mean")) / torch.sqrt(self.g(p + "batch_norm.running_var") + 1e-5)
            z = z * self.g(p + "batch_norm.weight") + self.g(p + "batch_norm.bias")
        return self.lin(z * torch.sigmoid(z), p + "pointwise_conv2.weight", p + "pointwise_conv2.bias")

    def ffn(self, x, name):
        h = self.lin(x, name + ".linear1.weight", name + ".linear1.bias")
        return self.lin(h * torch.sigmoid(h), name + ".linear2.weight", name + ".linear2.bias")

    def layer(self, i, x, pe, valid):
        p = "encoder.layers.%d." % i
        x = x + 0.5 * self.ffn(self.ln(x, p + "norm_feed_forward1"), p + "feed_forward1")
        x = x + self.attention(i, self.ln(x, p + "norm_self_att"), pe, valid)
        x = x + self.conv(i, self.ln(x, p + "norm_conv"), valid)
        x = x + 0.5 * self.ffn(self.ln(x, p + "norm_feed_forward2"), p + "feed_forward2")
        return self.ln(x, p + "norm_out")

    def encoder(self, mel, lens):
        x, v = self.sub(mel, lens)
        pe = _pos_table(x.shape[1], x.shape[2])
        for i in range(self.c.n_layers):
            x = self.layer(i, x, pe, v)
        return x


def _pos_table(T, D):
    pos = torch.arange(T - 1, -T, -1, dtype=F64, device="cuda")[:, None]
    ang = pos * torch.exp(torch.arange(0, D, 2, dtype=F64, device="cuda") * (-math.log(10000.0) / D))
    return torch.stack([torch.sin(ang), torch.cos(ang)], -1).reshape(2 * T - 1, D)


def _exact_mel(case, seed):
    pcm, lens = _pcm(case, seed)
    c = pm.Config(n_mels=case["n_mels"])
    T = 1 + case["samples"] // HOP
    off = (c.n_fft - c.win_length) // 2
    win = torch.zeros(c.n_fft, dtype=F64, device="cuda")
    win[off:off + c.win_length] = torch.from_numpy(pm.hann_window(c.win_length)).cuda().double()
    fb = torch.from_numpy(pm.mel_filterbank(c.sample_rate, c.n_fft, c.n_mels)).cuda().double()
    out = torch.zeros((case["B"], c.n_mels, T), dtype=F64, device="cuda")
    pre = float(np.float32(c.preemph))
    for b in range(case["B"]):
        n = int(lens[b])
        x = pcm[b, :n].double()
        x = torch.cat([x[:1], x[1:] - pre * x[:-1]])
        x = torch.nn.functional.pad(x, (c.n_fft // 2, c.n_fft // 2))
        f = x.unfold(0, c.n_fft, HOP) * win
        p = torch.fft.rfft(f).abs() ** 2
        y = torch.log(p @ fb.t() + c.log_zero_guard).t()
        v = n // HOP
        mu = y[:, :v].mean(1, keepdim=True)
        sd = y[:, :v].std(1, keepdim=True, unbiased=True)
        out[b, :, :v] = ((y - mu) / (sd + 1e-5))[:, :v]
    return out


def _exact_greedy(case, seed):
    m = _host_model(_model_key(case))
    lens = _lengths(case, seed, case["T"])
    g = lambda n: _dequant(m.tensors[n])  # noqa: E731
    H, L, B, D = m.cfg.pred_hidden, m.cfg.pred_rnn_layers, case["B"], m.cfg.d_model
    enc = _randn(seed, 6, B, case["T"], D).double() @ g("joint.enc.weight").t() + g("joint.enc.bias")
    pre = "decoder.prediction.dec_rnn.lstm."
    lstm = [[g(pre + "%s_l%d" % (n, i)) for n in ("weight_ih", "weight_hh", "bias_ih", "bias_hh")] for i in range(L)]
    wp, bp = g("joint.pred.weight"), g("joint.pred.bias")
    wo, bo, emb = g("joint.joint_net.2.weight"), g("joint.joint_net.2.bias"), g("decoder.prediction.embed.weight")
    n_tok, blank = m.cfg.vocab_size + 1, m.cfg.vocab_size
    x = torch.zeros((B, H), dtype=F64, device="cuda")
    h = [torch.zeros_like(x) for _ in range(L)]
    c = [torch.zeros_like(x) for _ in range(L)]
    t, sym, conf = [0] * B, [0] * B, [[] for _ in range(B)]
    while any(t[b] < lens[b] for b in range(B)):
        inp, nh, nc = x, [], []
        for i, (wi, wh, bi, bh) in enumerate(lstm):
            zi, zf, zg, zo = (inp @ wi.t() + h[i] @ wh.t() + bi + bh).chunk(4, 1)
            nc.append(torch.sigmoid(zf) * c[i] + torch.sigmoid(zi) * torch.tanh(zg))
            inp = torch.sigmoid(zo) * torch.tanh(nc[-1])
            nh.append(inp)
        at = torch.tensor([min(t[b], case["T"] - 1) for b in range(B)], device="cuda")
        z = torch.relu(enc[torch.arange(B, device="cuda"), at] + inp @ wp.t() + bp) @ wo.t() + bo
        tok = z[:, :n_tok].argmax(1)
        dur = z[:, n_tok:].argmax(1).tolist()
        pr = torch.softmax(z[:, :n_tok], 1).amax(1).tolist()
        live = [t[b] < lens[b] for b in range(B)]
        ids = tok.tolist()
        emit = torch.tensor([live[b] and ids[b] != blank for b in range(B)], device="cuda")[:, None]
        x = torch.where(emit, emb[tok], x)
        h = [torch.where(emit, a, b) for a, b in zip(nh, h)]
        c = [torch.where(emit, a, b) for a, b in zip(nc, c)]
        for b in range(B):
            if not live[b]:
                continue
            if ids[b] != blank:
                conf[b].append((n_tok * pr[b] - 1) / (n_tok - 1))
            sym[b] += 1
            t[b] += dur[b]
            if not (dur[b] == 0 and sym[b] < 10):
                t[b] += sym[b] == 10
                sym[b] = 0
    rect = np.zeros((B, 10 * case["T"]), np.float64)
    for b, v in enumerate(conf):
        rect[b, :len(v)] = v
    return [None, None, rect, None]


def exact(case, seed):
    k = case["kind"]
    if k == "mel":
        return _exact_mel(case, seed)
    if k == "greedy":
        return _exact_greedy(case, seed)
    e = _Exact(_model_key(case))
    if k == "stream":
        audio = _windows(case, seed, e.c.n_mels)
        outs = []
        for a in audio.split(16):
            n = a.shape[2]
            outs.append(e.encoder(a, np.full(a.shape[0], n, np.int64))[:, -2:])
        return torch.cat(outs)
    D = e.c.d_model
    if k in ("layer", "attn"):
        x = _randn(seed, 5, case["B"], case["T"], D).double()
        pe, lens = _pos_table(case["T"], D).float().double(), _lengths(case, seed, case["T"])
        return e.layer(0, x, pe, lens) if k == "layer" else e.attention(0, x, pe, lens)
    mel, lens = _features(case, seed, e.c.n_mels)
    if k == "sub":
        return e.sub(mel, lens - 1)[0]
    x = e.encoder(mel, lens - 1)
    z = e.lin(x, "ctc_decoder.decoder_layers.0.weight", "ctc_decoder.decoder_layers.0.bias")
    return [x, torch.log_softmax(z, -1)]
