"""The calls whose speed is measured: the stages of a transcription service as its programs call them, over the sizes
that they meet, from one short utterance to a full batch.

A case's "kind" names the stage:

  features  Features(extractor)(pieces): normalised log-mel features of audio pieces held on the GPU
  stem      SubsamplingStem(module)(features, frames): the encoder's 8x subsampling front end
  layers    EncoderLayers(blocks, ...)(x, lengths, meta): FastConformer layers over packed frames, W8A8 (with the
            feed-forward's second linear or both 2:4 sparse) or bf16, 8 or 16 heads
  linears   quantize_activations and Int8Linear, up (1280 -> 5120) then down (5120 -> 1280), with bias, dense or 2:4
  cross     StreamDecoder.fill_cross: the cross-attention keys and values of encoded pieces into their slots
  decode    StreamDecoder.set_active and step: four decoding steps of the active rows (one chunk)

Pieces: `pieces` of them, their lengths evenly spread from `shortest` to `longest`, the long ones between the short
ones. Lengths count samples (features), mel frames (stem) or encoder frames (layers, cross; 80 ms each).
"""

from __future__ import annotations

import math
import os
import random
import sys
import types

import numpy as np
import torch

sys.path.insert(1, os.path.join(os.getcwd(), "cohere-inference_amd"))

from kernels.fast_encoder import (EncoderLayers, Int8Linear, SubsamplingStem, metadata,  # noqa: E402
                                  quantize_activations)
from kernels.features import Features  # noqa: E402
from kernels.stream_decoder import StreamDecoder  # noqa: E402

D, FF, MELS, SUB = 1280, 5120, 128, 256  # encoder width, feed-forward width, mel bands, subsampling channels
DD, DFF, DHEADS, DLAYERS, VOCAB = 1024, 4096, 8, 8, 16384  # decoder
RATE, HOP, NFFT, WIN = 16000, 160, 512, 400
AUDIO_FRAMES, CACHE, STEPS = 376, 456, 4  # encoder frames of a 30 s piece, positions of a decoder slot, steps a pass
BF = torch.bfloat16


def listed() -> list[dict]:
    return [
        # eight requests of mixed length arriving together: the front end of one encoder chunk of a service
        dict(name="features_8_mixed", kind="features", pieces=8, shortest=2 * RATE + 77, longest=30 * RATE),
        # the same chunk through the subsampling stem: 8 pieces of 30 s (the service's 3000-frame chunk)
        dict(name="stem_8x30s", kind="stem", pieces=8, shortest=3001, longest=3001),
        # one two-second utterance alone (a voice command): latency and launches count
        dict(name="layers_int8_1x2s", kind="layers", pieces=1, shortest=26, longest=26, blocks=2, heads=16, int8=True,
             sparse=True, sparse_w1=False),
        # one 30 s clip alone: the lightly loaded service
        dict(name="layers_int8_1x30s", kind="layers", pieces=1, shortest=376, longest=376, blocks=2, heads=8,
             int8=True, sparse=True, sparse_w1=False),
        # the service's encoder chunk, 8 x 375 frames with both feed-forward linears 2:4 (the benchmark's block)
        dict(name="layers_int8_8x30s", kind="layers", pieces=8, shortest=375, longest=375, blocks=1, heads=16,
             int8=True, sparse=True, sparse_w1=True),
        # a whole batch in one encoder call, clips of 12 to 30 s
        dict(name="layers_int8_32_mixed", kind="layers", pieces=32, shortest=150, longest=376, blocks=1, heads=16,
             int8=True, sparse=True, sparse_w1=True),
        # the default encoder (bf16 weights, 8 heads) over a chunk of mixed clips
        dict(name="layers_bf16_8_mixed", kind="layers", pieces=8, shortest=97, longest=376, blocks=1, heads=8,
             int8=False, sparse=False, sparse_w1=False),
        # the benchmark's pair of 2:4 linears with bias at 8 x 375 rows, activations quantized per row
        dict(name="linears_24_3000", kind="linears", rows=3000, sparse=True),
        # the encoded chunk handed to the decoder: 8 clips' cross-attention keys and values into int8 caches
        dict(name="cross_8x30s", kind="cross", pieces=8, shortest=375, longest=375, int8=True),
        # one request decoding alone: the smallest step
        dict(name="decode_int8_1", kind="decode", rows=1, shortest=120, longest=120, int8=True),
        # a full decoder, 64 rows at mixed positions (the benchmark's step)
        dict(name="decode_int8_64", kind="decode", rows=64, shortest=1, longest=440, int8=True),
        # the default decoder (bf16 weights and caches) under moderate load
        dict(name="decode_bf16_24", kind="decode", rows=24, shortest=8, longest=300, int8=False),
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng: random.Random) -> dict:
    kind = rng.choice(["features", "stem", "layers", "layers", "layers", "linears", "cross", "decode", "decode"])
    if kind in ("features", "stem"):
        n = _log_int(rng, 1, 16)
        lo, hi = ((RATE // 2, 30 * RATE) if kind == "features" else (50, 3001))
        a, b = sorted(_log_int(rng, lo, hi) for _ in range(2))
        return dict(kind=kind, pieces=n, shortest=a, longest=b)
    if kind in ("layers", "cross"):
        n = _log_int(rng, 1, 24 if kind == "layers" else 8)
        a, b = sorted(_log_int(rng, 6, 376) for _ in range(2))
        if kind == "cross":
            return dict(kind=kind, pieces=n, shortest=a, longest=b, int8=rng.random() < 0.7)
        int8 = rng.random() < 0.75
        sparse = int8 and rng.random() < 0.8
        return dict(kind=kind, pieces=n, shortest=a, longest=b, blocks=1, heads=rng.choice([8, 16]), int8=int8,
                    sparse=sparse, sparse_w1=sparse and rng.random() < 0.5)
    if kind == "linears":
        return dict(kind=kind, rows=_log_int(rng, 16, 6000), sparse=rng.random() < 0.6)
    a, b = sorted(rng.randint(1, 448) for _ in range(2))
    return dict(kind=kind, rows=_log_int(rng, 1, 64), shortest=a, longest=b, int8=rng.random() < 0.7)


def _spread(n: int, lo: int, hi: int) -> list[int]:
    """n whole numbers evenly from lo to hi, in an order that mixes short and long."""
    v = [lo + (hi - lo) * i // max(n - 1, 1) for i in range(n)] if n > 1 else [hi]
    return v[::2] + v[1::2][::-1]


def _lengths(case: dict) -> list[int]:
    return _spread(case["pieces"], case["shortest"], case["longest"])


# ---- inputs, from the seed alone -------------------------------------------------------------------------------------

class _Draw:
    """Random tensors on the GPU from one generator."""

    def __init__(self, seed: int):
        self.dev = torch.device("cuda")
        self.g = torch.Generator(device=self.dev).manual_seed(seed)

    def normal(self, *shape, std=1.0, mean=0.0, dtype=BF):
        return (mean + std * torch.randn(*shape, generator=self.g, device=self.dev)).to(dtype)

    def uniform(self, *shape, lo=0.0, hi=1.0, dtype=torch.float32):
        return (lo + (hi - lo) * torch.rand(*shape, generator=self.g, device=self.dev)).to(dtype)

    def xavier(self, n, k, pruned=False):
        a = math.sqrt(6.0 / (n + k))
        w = self.uniform(n, k, lo=-a, hi=a, dtype=BF)
        return self.prune(w) if pruned else w

    def prune(self, w):
        """Two random positions of every four along K zero, as calibrated 2:4 weights arrive."""
        keep = torch.rand(w.shape[0], w.shape[1] // 4, 4, generator=self.g, device=self.dev).argsort(-1) < 2
        return torch.where(keep.reshape(w.shape), w, torch.zeros((), dtype=BF, device=self.dev))

    def ints(self, lo, hi, *shape, dtype=torch.int64):
        return torch.randint(lo, hi, shape, generator=self.g, device=self.dev, dtype=dtype)

    def linear(self, n, k, pruned=False):
        return types.SimpleNamespace(weight=self.xavier(n, k, pruned), bias=self.normal(n, std=0.05))

    def norm(self, n):
        return types.SimpleNamespace(weight=self.normal(n, std=0.1, mean=1.0), bias=self.normal(n, std=0.05), eps=1e-5)


def _block(r: _Draw, heads: int, prune_w1: bool, prune_w2: bool):
    """A FastConformer block with the attributes EncoderLayers reads (random weights, 1280 wide)."""
    ns = types.SimpleNamespace
    ff = lambda: ns(linear1=r.linear(FF, D, prune_w1), linear2=r.linear(D, FF, prune_w2))  # noqa: E731
    att = ns(q_proj=r.linear(D, D), k_proj=r.linear(D, D), v_proj=r.linear(D, D), o_proj=r.linear(D, D),
             bias_u=r.normal(heads, D // heads, std=0.2), bias_v=r.normal(heads, D // heads, std=0.2),
             relative_k_proj=ns(weight=r.xavier(D, D)))
    pw1, pw2 = r.linear(2 * D, D), r.linear(D, D)
    pw1.weight, pw2.weight = pw1.weight[:, :, None], pw2.weight[:, :, None]
    dw = ns(weight=r.normal(D, 1, 9, std=0.3), bias=r.normal(D, std=0.05), in_channels=D)
    bn = ns(weight=r.normal(D, std=0.1, mean=1.0), bias=r.normal(D, std=0.05),
            running_mean=r.normal(D, std=0.05), running_var=r.uniform(D, lo=1.0, hi=1.2, dtype=BF), eps=1e-5)
    return ns(feed_forward1=ff(), self_attn=att, conv=ns(pointwise_conv1=pw1, depthwise_conv=dw, norm=bn,
                                                          pointwise_conv2=pw2), feed_forward2=ff(),
              norm_feed_forward1=r.norm(D), norm_self_att=r.norm(D), norm_conv=r.norm(D), norm_feed_forward2=r.norm(D),
              norm_out=r.norm(D))


def _inv_freq():
    return 1.0 / (10000.0 ** (torch.arange(0, D, 2, dtype=torch.float) / D))


def _layer_inputs(case, seed):
    r = _Draw(seed)
    blocks = [_block(r, case["heads"], case["sparse_w1"], case["sparse"]) for _ in range(case["blocks"])]
    return blocks, r.normal(sum(_lengths(case)), D)


def _mel_filters() -> torch.Tensor:
    """128 triangular bands on Slaney's mel scale over the 257 bins, with Slaney's area normalisation."""
    step = math.log(6.4) / 27.0
    to_mel = lambda f: f * 3 / 200 if f < 1000 else 15.0 + math.log(f / 1000.0) / step  # noqa: E731
    mels = np.linspace(0.0, to_mel(RATE / 2), MELS + 2)
    hz = np.where(mels < 15.0, mels * 200 / 3, 1000.0 * np.exp(step * (mels - 15.0)))
    bins = np.linspace(0, RATE / 2, NFFT // 2 + 1)
    up = (bins[None] - hz[:-2, None]) / (hz[1:-1] - hz[:-2])[:, None]
    down = (hz[2:, None] - bins[None]) / (hz[2:] - hz[1:-1])[:, None]
    w = np.maximum(0, np.minimum(up, down)) * (2.0 / (hz[2:] - hz[:-2]))[:, None]
    return torch.from_numpy(w.astype(np.float32))


def _audio(case, seed):
    """Per piece a noise floor and a few tones that start and stop, fp32 at about -20 dBFS."""
    r = _Draw(seed)
    out = []
    for n in _lengths(case):
        t = torch.arange(n, device=r.dev, dtype=torch.float64) / RATE
        x = 0.03 * torch.randn(n, generator=r.g, device=r.dev, dtype=torch.float64)
        for _ in range(4):
            f, ph, a, b = r.uniform(4, dtype=torch.float64)
            gate = torch.sin(2 * math.pi * (0.2 + 2 * a) * t + 6.28 * b) > 0
            x = x + 0.08 * gate * torch.sin(2 * math.pi * (100 + 2900 * f) * t + 6.28 * ph)
        out.append(x.float())
    return out


def _stem_inputs(case, seed):
    r = _Draw(seed)
    frames = _lengths(case)

    def conv(cin, cout, k, groups):
        c = torch.nn.Conv2d(cin, cout, k, stride=2 if k == 3 else 1, padding=k // 2, groups=groups, device="meta")
        c = c.to_empty(device=r.dev)
        fan = cin // groups * k * k
        c.weight.data.copy_(r.normal(*c.weight.shape, std=fan ** -0.5, dtype=torch.float32))
        c.bias.data.copy_(r.normal(*c.bias.shape, std=0.05, dtype=torch.float32))
        return c.to(BF)

    layers = [conv(1, SUB, 3, 1), conv(SUB, SUB, 3, SUB), conv(SUB, SUB, 1, 1), conv(SUB, SUB, 3, SUB),
              conv(SUB, SUB, 1, 1)]
    lin = r.linear(D, SUB * MELS // 8)
    lin.in_features = SUB * MELS // 8
    feats = torch.zeros(len(frames), max(frames), MELS, device=r.dev, dtype=BF)
    for i, f in enumerate(frames):
        feats[i, :f] = r.normal(f, MELS)
    return types.SimpleNamespace(layers=layers, linear=lin), feats, frames


def _linear_inputs(case, seed):
    r = _Draw(seed)
    x = r.normal(case["rows"], D)
    up, down = r.normal(FF, D, std=0.02), r.normal(D, FF, std=0.02)
    if case["sparse"]:
        up, down = r.prune(up), r.prune(down)
    return x, up, r.normal(FF, std=0.01), down, r.normal(D, std=0.01)


def _decoder_model(r: _Draw):
    """A decoder with the attributes StreamDecoder reads (random weights: 8 layers, 1024 wide, vocabulary 16384)."""
    ns = types.SimpleNamespace

    def lin(n, k):
        return ns(weight=r.normal(n, k, std=k ** -0.5), bias=r.normal(n, std=0.05))

    att = lambda: ns(q_proj=lin(DD, DD), k_proj=lin(DD, DD), v_proj=lin(DD, DD), o_proj=lin(DD, DD))  # noqa: E731
    layers = [ns(self_attn=att(), encoder_attn=att(), mlp=ns(fc1=lin(DFF, DD), fc2=lin(DD, DFF)),
                 input_layernorm=r.norm(DD), post_attention_layernorm=r.norm(DD), final_layernorm=r.norm(DD))
              for _ in range(DLAYERS)]
    proj = lin(DD, D)
    dec = ns(layers=layers, embed_tokens=ns(weight=r.normal(VOCAB, DD)), pos_emb=ns(weight=r.normal(512, DD, std=0.5)),
             embedding_layernorm=r.norm(DD), norm=r.norm(DD), proj=proj)
    cfg = ns(num_attention_heads=DHEADS, hidden_size=DD, head_dim=DD // DHEADS, eos_token_id=3, pad_token_id=2)
    return ns(model=ns(decoder=dec), proj_out=lin(VOCAB, DD), config=cfg)


def _bucket(rows: int) -> int:
    return next(b for b in StreamDecoder.BUCKETS if b >= rows)


def _decode_inputs(case, seed):
    """The model, the slots' tokens, positions and audio lengths, and the caches' contents, one tensor each:
    (layer, slot, head, position, 128), int8 values with a scale per vector, or bf16."""
    r = _Draw(seed)
    model = _decoder_model(r)
    rows = case["rows"]
    tokens = r.ints(4, VOCAB, rows, CACHE)
    pos = torch.tensor(_spread(rows, case["shortest"], case["longest"]), device=r.dev)
    audio = r.ints(AUDIO_FRAMES // 3, AUDIO_FRAMES + 1, rows)
    caches = []
    for length in (CACHE + 9, CACHE + 9, AUDIO_FRAMES, AUDIO_FRAMES):
        shape = (DLAYERS, rows, DHEADS, length)
        if case["int8"]:
            caches.append((r.ints(-127, 128, *shape, DD // DHEADS, dtype=torch.int8),
                           r.uniform(*shape, lo=0.01, hi=0.03)))
        else:
            caches.append((r.normal(*shape, DD // DHEADS), None))
    return model, tokens, pos, audio, caches


# ---- what a program has in hand, and one pass ------------------------------------------------------------------------

@torch.no_grad()
def prepare(case: dict, seed: int):
    kind, s = case["kind"], types.SimpleNamespace(kind=case["kind"])
    if kind == "features":
        ext = types.SimpleNamespace(n_fft=NFFT, hop_length=HOP, win_length=WIN, preemphasis=0.97,
                                    mel_filters=_mel_filters())
        s.features, s.pieces = Features(ext), _audio(case, seed)
    elif kind == "stem":
        sub, s.feats, s.frames = _stem_inputs(case, seed)
        s.stem = SubsamplingStem(sub)
    elif kind == "layers":
        blocks, s.x = _layer_inputs(case, seed)
        s.layers = EncoderLayers(blocks, _inv_freq(), sparse=case["sparse"], sparse_w1=case["sparse_w1"],
                                 int8=case["int8"])
        s.lengths = _lengths(case)
        s.meta = metadata(s.lengths, s.x.device)
    elif kind == "linears":
        s.x, up, bu, down, bd = _linear_inputs(case, seed)
        s.up, s.down = Int8Linear(up, bu, sparse=case["sparse"]), Int8Linear(down, bd, sparse=case["sparse"])
    elif kind == "cross":
        r = _Draw(seed)
        s.lengths = _lengths(case)
        s.dec = StreamDecoder(_decoder_model(r), slots=len(s.lengths), max_prompt=4, max_new_tokens=4, buckets=(1,),
                              int8=case["int8"], frames=AUDIO_FRAMES, capture=False)
        s.hidden = r.normal(sum(s.lengths), D)
        s.slots = list(range(len(s.lengths)))[::-1]
    else:
        model, tokens, pos, audio, caches = _decode_inputs(case, seed)
        rows = case["rows"]
        s.rows = rows
        s.dec = dec = StreamDecoder(model, slots=max(rows, _bucket(rows)), max_prompt=CACHE, max_new_tokens=8,
                                    buckets=(_bucket(rows),), int8=case["int8"], frames=AUDIO_FRAMES, chunk=STEPS,
                                    capture=False)
        # the step's graphs are recorded once the decoder's buffers are filled: recording runs every launch once on the
        # decoder's own stream, which does not wait for the fills queued on this one
        torch.cuda.synchronize()
        dec._capture()
        s.slots = list(range(rows))
        # the rows' texts so far, and the steps' tokens: given, so that a pass does the same work every time
        dec.admit(s.slots, list(tokens.cpu()), audio.tolist())
        dec.stream.synchronize()
        for (q, sc), to, to_s in zip(caches, (dec.self_k, dec.self_v, dec.cross_k, dec.cross_v),
                                     (dec.self_ks, dec.self_vs, dec.cross_ks, dec.cross_vs)):
            to[:, :rows].copy_(q)
            if sc is not None:
                to_s[:, :rows].copy_(sc)
        s.pos = pos.to(torch.int32)
        s.tok = tokens.gather(1, pos[:, None])[:, 0].contiguous()
    torch.cuda.synchronize()
    return s


@torch.no_grad()
def run(s):
    if s.kind == "features":
        feats, frames = s.features(s.pieces)
        return {"features": feats, "frames": frames}
    if s.kind == "stem":
        x, lengths = s.stem(s.feats, s.frames)
        return {"x": x, "lengths": lengths}
    if s.kind == "layers":
        return s.layers(s.x.clone(), s.lengths, s.meta)
    if s.kind == "linears":
        y = s.up(*quantize_activations(s.x))
        return {"up": y, "down": s.down(*quantize_activations(y))}
    if s.kind == "cross":
        d = s.dec
        d.fill_cross(s.hidden, s.lengths, s.slots)
        return [t for t in (d.cross_k, d.cross_v, d.cross_ks, d.cross_vs) if t is not None]
    d, here = s.dec, torch.cuda.current_stream()
    d.stream.wait_stream(here)
    with torch.cuda.stream(d.stream):  # the rows back where they were
        d.pos[:s.rows].copy_(s.pos)
        d.tok[:s.rows].copy_(s.tok)
    d.step(d.set_active(s.slots), STEPS)
    here.wait_stream(d.stream)  # the logits are read on the caller's stream
    return {"logits": d.logits[:s.rows], "pos": d.pos[:s.rows]}


# ---- what a pass cannot do without -----------------------------------------------------------------------------------

def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "features":
        n = sum(_lengths(case))
        frames = n // HOP
        return {"bytes": 4 * n + 2 * MELS * frames, "flops": frames * (5 * NFFT / 2 * math.log2(NFFT) + 4 * NFFT)}
    if kind == "stem":
        f = sum(_lengths(case))
        out = f / 8
        rows2, rows4 = f / 4 * 32, f / 8 * 16  # positions after the first and second stage
        flops = 2 * (f / 2 * 64 * SUB * 9 + rows2 * SUB * (9 + SUB) + rows4 * SUB * (9 + SUB) + out * 4096 * D)
        return {"bytes": 2 * (f * MELS + out * D + 4096 * D + 2 * SUB * SUB), "flops": flops}
    if kind == "layers":
        lens = _lengths(case)
        m, b = sum(lens), case["blocks"]
        one, sp = (1.0, 0.625) if case["int8"] else (2.0, 0.0)  # bytes a weight, dense and 2:4
        keep = lambda on: 0.5 if on else 1.0  # noqa: E731
        dense = D * 3 * D + D * D + 2 * D * D + D * D
        w1, w2 = 2 * D * FF, 2 * D * FF
        weights = one * dense + (sp if case["sparse_w1"] else one) * w1 + (sp if case["sparse"] else one) * w2
        macs = m * (dense + keep(case["sparse_w1"]) * w1 + keep(case["sparse"]) * w2 + 9 * D)
        macs += sum(3 * n * n * D for n in lens)
        table = 2 * D * sum({min(2 * n + 62, 1087) for n in [max(lens)]})
        return {"bytes": b * (weights + table + 2 * m * D * 2), "flops": b * 2.0 * macs}
    if kind == "linears":
        m, sp = case["rows"], case["sparse"]
        return {"bytes": 2 * m * (D + FF + D) + 2 * D * FF * (0.625 if sp else 1.0),
                "flops": 2.0 * 2 * m * D * FF * (0.5 if sp else 1.0)}
    if kind == "cross":
        m = sum(_lengths(case))
        n = 2 * DLAYERS * DD
        return {"bytes": 2 * (m * D + D * DD + n * DD) + m * n * (1 if case["int8"] else 2),
                "flops": 2.0 * m * (D * DD + DD * n)}
    rows = case["rows"]
    one = 1 if case["int8"] else 2
    big = DLAYERS * (3 * DD * DD + 2 * DD * DFF) + VOCAB * DD  # int8 weights when int8
    small = DLAYERS * 3 * DD * DD  # the attention outputs and the cross-attention query stay bf16
    ctx = sum(_spread(rows, case["shortest"], case["longest"])) + rows * AUDIO_FRAMES * 2 / 3
    kv = DLAYERS * 2 * DD * ctx
    return {"bytes": STEPS * (one * big + 2 * small + one * kv),
            "flops": STEPS * 2.0 * (rows * (big + small) + 2 * kv / 2 * 2)}


# ---- how far another correct implementation may be off ---------------------------------------------------------------

def tolerance(case: dict):
    """Measured against other summation orders and exact(): about four times what those show."""
    kind = case["kind"]
    if kind == "features":  # fp32 spectrum and logarithm, bf16 out
        return {"rel": 2e-3, "max": 2e-2}
    if kind == "stem":  # bf16 convolutions and products
        return {"rel": 6e-3, "max": 5e-2}
    if kind == "layers":  # a rounding that moves an int8 activation by one step travels through the block
        if case["int8"]:
            return {"rel": 8e-3, "max": 0.25} if case["blocks"] == 1 else {"rel": 2e-2, "max": 0.4}
        return {"rel": 1.2e-2, "max": 0.15}
    if kind == "linears":  # exact integer sums; the second linear's int8 inputs move by a step
        return {"rel": 4e-3, "max": 5e-2}
    if kind == "cross":
        return {"rel": 4e-3, "max": 5e-2, "differ": 0.01}
    return {"rel": 3e-2, "max": 0.3}  # eight layers in bf16, int8 caches


# ---- the same in 64 bits ---------------------------------------------------------------------------------------------

def _f8(t):
    return t.double()


def _weight_q8(w):
    """A weight as its symmetric int8 rows say it: round(w / s) s with s = fp32(amax) fp32(1 / 127)."""
    w = w.float()
    s = w.abs().amax(-1, keepdim=True).clamp_min(1e-12) * float(np.float32(1) / np.float32(127))
    return torch.round(w / s).clamp(-127, 127).double() * s.double()


def _rows_q8(h, group=None):
    """Activations as their int8 rows (or groups of columns) say them."""
    v = h.reshape(h.shape[0], -1, group or h.shape[1])
    s = v.abs().amax(-1, keepdim=True) / 127
    s = torch.where(s > 0, s, torch.ones_like(s))
    return (torch.round(v / s) * s).reshape(h.shape)


def _ln(x, m):
    return torch.nn.functional.layer_norm(x, (x.shape[-1],), _f8(m.weight), _f8(m.bias), m.eps)


def _exact_block(x, blk, lens, heads, int8, table, off):
    wq = _weight_q8 if int8 else _f8
    act = _rows_q8 if int8 else (lambda h, group=None: h)
    lin = lambda h, m, group=None: act(h, group) @ wq(m.weight.flatten(1)).T + _f8(m.bias)  # noqa: E731

    def ff(x, norm, f):
        t = lin(_ln(x, norm), f.linear1)
        return x + 0.5 * lin(t * torch.sigmoid(t), f.linear2, 256)

    x = ff(x, blk.norm_feed_forward1, blk.feed_forward1)
    at, d = blk.self_attn, D // heads
    h = act(_ln(x, blk.norm_self_att))
    q, k, v = (h @ wq(m.weight).T + _f8(m.bias) for m in (at.q_proj, at.k_proj, at.v_proj))
    rk = (table @ _f8(at.relative_k_proj.weight).T).view(-1, heads, d)
    out, s0 = torch.empty_like(x), 0
    for n in lens:
        qs, ks, vs = (t[s0:s0 + n].view(n, heads, d).transpose(0, 1) for t in (q, k, v))
        i = torch.arange(n, device=x.device)
        sc = (qs + _f8(at.bias_u)[:, None]) @ ks.transpose(1, 2)
        p = (qs + _f8(at.bias_v)[:, None]) @ rk[off - (n - 1):off + n].permute(1, 2, 0)
        sc = sc + p.gather(2, (i[:, None] - i[None] + n - 1).expand(heads, n, n))
        out[s0:s0 + n] = (torch.softmax(sc * d ** -0.5, -1) @ vs).transpose(0, 1).reshape(n, D)
        s0 += n
    x = x + lin(out, at.o_proj)
    cv = blk.conv
    h = lin(_ln(x, blk.norm_conv), cv.pointwise_conv1)
    h = h[:, :D] * torch.sigmoid(h[:, D:])
    bn, w = cv.norm, _f8(cv.depthwise_conv.weight[:, 0])
    y, s0 = torch.empty_like(h), 0
    for n in lens:
        pad = torch.nn.functional.pad(h[s0:s0 + n], (0, 0, 4, 4))
        y[s0:s0 + n] = sum(pad[t:t + n] * w[:, t] for t in range(9))
        s0 += n
    y = y + _f8(cv.depthwise_conv.bias)
    y = (y - _f8(bn.running_mean)) * _f8(bn.weight) / torch.sqrt(_f8(bn.running_var) + bn.eps) + _f8(bn.bias)
    x = x + lin(y * torch.sigmoid(y), cv.pointwise_conv2)
    x = ff(x, blk.norm_feed_forward2, blk.feed_forward2)
    return _ln(x, blk.norm_out)


def _exact_layers(case, seed):
    blocks, x = _layer_inputs(case, seed)
    lens = _lengths(case)
    d = torch.arange(-511, 512 + 64, device=x.device, dtype=torch.float64)
    fr = d[:, None] * _f8(_inv_freq().to(x.device))
    table = _f8(torch.stack([fr.sin(), fr.cos()], -1).reshape(len(d), -1).to(BF))
    x = _f8(x)
    for b in blocks:
        x = _exact_block(x, b, lens, case["heads"], case["int8"], table, 511)
    return x


def _exact_features(case, seed):
    dev = torch.device("cuda")
    mel = _f8(_mel_filters()).to(dev)
    win = torch.zeros(NFFT, dtype=torch.float64, device=dev)
    win[(NFFT - WIN) // 2:(NFFT + WIN) // 2] = torch.hann_window(WIN, periodic=False, dtype=torch.float64, device=dev)
    lens = _lengths(case)
    out = torch.zeros(len(lens), max(lens) // HOP + 1, MELS, dtype=torch.float64, device=dev)
    for b, x in enumerate(_audio(case, seed)):
        x = _f8(x)
        n = len(x) // HOP
        x = torch.cat([x[:1], x[1:] - 0.97 * x[:-1]])
        fr = torch.nn.functional.pad(x, (NFFT // 2, NFFT // 2 + HOP)).unfold(0, NFFT, HOP)[:n]
        lm = torch.log((torch.fft.rfft(fr * win).abs() ** 2) @ mel.T + 2.0 ** -24)
        out[b, :n] = (lm - lm.mean(0)) / (lm.std(0) + 1e-5)
    return {"features": out, "frames": [None] * len(lens)}


def _exact_stem(case, seed):
    sub, feats, frames = _stem_inputs(case, seed)
    full, dw1, pw1, dw2, pw2 = sub.layers

    def taps(h, c):
        """3x3, stride 2, padded by one: h (T, F, channels or 1) by one filter a channel."""
        h = torch.nn.functional.pad(h, (0, 0, 1, 1, 1, 1))
        t, f = (h.shape[0] - 1) // 2, (h.shape[1] - 1) // 2
        w = _f8(c.weight).flatten(1)
        return sum(h[i:i + 2 * t - 1:2, j:j + 2 * f - 1:2] * w[:, 3 * i + j] for i in range(3) for j in range(3)) \
            + _f8(c.bias)

    point = lambda h, c: torch.relu(h @ _f8(c.weight).flatten(1).T + _f8(c.bias))  # noqa: E731
    out = []
    for b, n in enumerate(frames):
        h = torch.relu(taps(_f8(feats[b, :n, :, None]), full))
        h = point(taps(h, dw1), pw1)
        h = point(taps(h, dw2), pw2)
        out.append(h.transpose(1, 2).flatten(1) @ _f8(sub.linear.weight).T + _f8(sub.linear.bias))
    return {"x": torch.cat(out), "lengths": [None] * len(frames)}


def _exact_cross(case, seed):
    r = _Draw(seed)
    model = _decoder_model(r)
    lens = _lengths(case)
    h = _f8(r.normal(sum(lens), D))
    dec = model.model.decoder
    h = h @ _f8(dec.proj.weight).T + _f8(dec.proj.bias)
    slots, S = list(range(len(lens)))[::-1], len(lens) + 1
    res = []
    for name in ("k_proj", "v_proj"):
        full = torch.zeros(DLAYERS, S, DHEADS, AUDIO_FRAMES, DD // DHEADS, dtype=torch.float64, device=h.device)
        for i, ly in enumerate(dec.layers):
            m = getattr(ly.encoder_attn, name)
            kv = h @ _f8(m.weight).T + _f8(m.bias)
            s0 = 0
            for sl, n in zip(slots, lens):
                full[i, sl, :, :n] = kv[s0:s0 + n].view(n, DHEADS, -1).transpose(0, 1)
                s0 += n
        res.append(full)
    if not case["int8"]:
        return res
    scale = lambda t: torch.where(t.abs().amax(-1) > 0, t.abs().amax(-1) / 127, 1.0)  # noqa: E731
    return [None, None, scale(res[0]), scale(res[1])]


def _exact_decode(case, seed):
    model, tokens, pos, audio, caches = _decode_inputs(case, seed)
    dec, int8, rows = model.model.decoder, case["int8"], case["rows"]
    wq = _weight_q8 if int8 else _f8
    (sk, sv, ck, cv) = [_f8(q) if sc is None else _f8(q) * _f8(sc)[..., None] for q, sc in caches]
    last = torch.arange(CACHE + 9, device=pos.device)
    heard = torch.arange(AUDIO_FRAMES, device=pos.device) < audio[:, None]
    lin = lambda h, m, w=_f8: h @ w(m.weight).T + _f8(m.bias)  # noqa: E731
    every = torch.arange(rows, device=pos.device)

    def attend(q, k, v, mask):
        sc = (k @ q[..., None])[..., 0] * (DD // DHEADS) ** -0.5
        p = torch.softmax(sc.masked_fill(~mask[:, None], -math.inf), -1)
        return (p[..., None, :] @ v)[..., 0, :].reshape(rows, DD)

    def kept(t):
        """What the int8 cache keeps of a new key or value."""
        return _rows_q8(t.reshape(-1, DD // DHEADS)).view_as(t) if int8 else t

    for step in range(STEPS):
        at = pos + step
        tok = tokens.gather(1, at[:, None])[:, 0]
        x = _ln(_f8(dec.embed_tokens.weight)[tok] + _f8(dec.pos_emb.weight)[at], dec.embedding_layernorm)
        for i, ly in enumerate(dec.layers):
            h = _ln(x, ly.input_layernorm)
            sa, ca = ly.self_attn, ly.encoder_attn
            q, k, v = (lin(h, m, wq).view(rows, DHEADS, -1) for m in (sa.q_proj, sa.k_proj, sa.v_proj))
            sk[i, every, :, at], sv[i, every, :, at] = k, v  # the new token's own as computed
            x = x + lin(attend(q, sk[i], sv[i], last <= at[:, None]), sa.o_proj)
            sk[i, every, :, at], sv[i, every, :, at] = kept(k), kept(v)
            q = lin(_ln(x, ly.post_attention_layernorm), ca.q_proj).view(rows, DHEADS, -1)
            x = x + lin(attend(q, ck[i], cv[i], heard), ca.o_proj)
            h = torch.relu(lin(_ln(x, ly.final_layernorm), ly.mlp.fc1, wq))
            x = x + lin(h, ly.mlp.fc2, wq)
    return {"logits": lin(_ln(x, dec.norm), model.proj_out, wq), "pos": None}


@torch.no_grad()
def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "linears":
        x, up, bu, down, bd = _linear_inputs(case, seed)
        y = _rows_q8(_f8(x)) @ _weight_q8(up).T + _f8(bu)
        return {"up": y, "down": _rows_q8(y) @ _weight_q8(down).T + _f8(bd)}
    return {"features": _exact_features, "stem": _exact_stem, "layers": _exact_layers, "cross": _exact_cross,
            "decode": _exact_decode}[kind](case, seed)
