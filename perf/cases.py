"""The framework's work as a user has it done, as cases that can be timed and checked.

A case is a dict of plain values.  listed() gives the named cases, draw(rng)
another one of the same ranges, prepare(case, seed) what a program has in hand
before the call (a loaded model or a layer's weights, inputs on the device),
run(state) one pass through the public entry points, work(case) the bytes and
operations that pass cannot do without, tolerance(case) what another correct
implementation of the same precision may differ by, and exact(case, seed) the
same outputs in 64 bits from plain torch.

Kinds of case:
  embed      PCM on the device -> speaker embeddings (voicedetect_gpu_embed_batch_async)
  analyze    PCM on the device -> wav2vec2 emotion logits (voicedetect_gpu_analyze_batch_async)
  fbank      PCM -> log-mel features and their per-clip means (vdk_fbank_ex)
  conv       one 3x3 layer of a residual encoder (vdk_conv2d_ex)
  attention  one wav2vec2 self-attention core (vdk_attention)
  asp        ECAPA's attentive statistics pooling (vdk_asp_attn_pool)
  identify   queries against an enrolled registry (vdk_registry_topk)
"""
import math
import os
import sys
import tempfile

import numpy as np
import torch
import torch.nn.functional as F

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "voice-detect.cpp_amd"))

from vdamd import gguf, lib, synth  # noqa: E402

SR = 16000
WIN, HOP, NFFT, MELS = 400, 160, 512, 80
DEV = "cuda"


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # one 3 s utterance to be verified: the reference's own unit of work, bound by latency
        {"name": "embed_resnet34_1x3s", "kind": "embed", "model": "resnet34", "batch": 1, "samples": 48000},
        # an enrolment job in bulk: the benchmark's headline workload
        {"name": "embed_resnet34_64x3s", "kind": "embed", "model": "resnet34", "batch": 64, "samples": 48000},
        # a few short utterances of an uneven length, as a voice-activity detector cuts them
        {"name": "embed_ecapa_5x2.61s", "kind": "embed", "model": "ecapa", "batch": 5, "samples": 41777},
        # the benchmark's CAM++ workload: q8_0 weights, 10 s clips
        {"name": "embed_campplus_32x10s", "kind": "embed", "model": "campplus", "batch": 32, "samples": 160000},
        # two speakers compared on one longer, odd-length recording each
        {"name": "embed_eres2net_2x7.3s", "kind": "embed", "model": "eres2net", "batch": 2, "samples": 116801},
        # emotion of one utterance (analyze of a single file)
        {"name": "analyze_emotion_1x3.2s", "kind": "analyze", "model": "emotion", "batch": 1, "samples": 51200},
        # the front end that every speaker model starts with, at the headline batch
        {"name": "fbank_64x3s", "kind": "fbank", "batch": 64, "samples": 48000},
        # the most frequent layer of the headline encoder, on 5 s clips (126 columns)
        {"name": "conv3x3_128_16x126", "kind": "conv", "batch": 16, "H": 20, "W": 126, "IC": 128, "OC": 128,
         "stride": 1},
        # wav2vec2-large attention on 10 s clips
        {"name": "attention_8x499", "kind": "attention", "batch": 8, "T": 499, "heads": 16},
        # ECAPA's pooling over a batch of 6.3 s clips
        {"name": "asp_pool_16x629", "kind": "asp", "batch": 16, "T": 629, "C": 1536},
        # one speaker looked up among a small team: the smallest call
        {"name": "identify_1x3000", "kind": "identify", "batch": 1, "rows": 3000, "dim": 256, "k": 5},
        # a batch looked up in a large registry (the benchmark's identify leg)
        {"name": "identify_64x100k", "kind": "identify", "batch": 64, "rows": 100000, "dim": 192, "k": 10},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        kind = rng.choice(["embed", "embed", "embed", "embed", "analyze", "fbank", "conv", "attention", "asp",
                           "identify", "identify"])
        if kind == "embed":
            c = {"kind": kind, "model": rng.choice(["resnet34", "ecapa", "campplus", "eres2net"]),
                 "batch": _log_int(rng, 1, 64), "samples": _log_int(rng, 1.0 * SR, 12.0 * SR)}
        elif kind == "analyze":
            c = {"kind": kind, "model": "emotion", "batch": _log_int(rng, 1, 32),
                 "samples": _log_int(rng, 1.0 * SR, 10.0 * SR)}
        elif kind == "fbank":
            c = {"kind": kind, "batch": _log_int(rng, 1, 64), "samples": _log_int(rng, 1.0 * SR, 20.0 * SR)}
        elif kind == "conv":
            stage = rng.choice([1, 2, 3])                      # 64, 128 or 256 channels
            oc, stride = 32 << stage, rng.choice([1, 1, 1, 2])  # a stage's first conv halves the map
            frames = _log_int(rng, 98, 1198)
            scale = 1 << (stage - (1 if stride == 2 else 0))
            c = {"kind": kind, "batch": _log_int(rng, 1, 64), "H": MELS // scale, "W": (frames - 1) // scale + 1,
                 "IC": oc // stride, "OC": oc, "stride": stride}
        elif kind == "attention":
            c = {"kind": kind, "batch": _log_int(rng, 1, 64), "T": _log_int(rng, 49, 749),
                 "heads": rng.choice([12, 16])}
        elif kind == "asp":
            c = {"kind": kind, "batch": _log_int(rng, 1, 64), "T": _log_int(rng, 98, 998),
                 "C": rng.choice([1536, 3072])}
        else:
            c = {"kind": kind, "batch": _log_int(rng, 1, 64), "rows": _log_int(rng, 100, 100000),
                 "dim": rng.choice([192, 256, 512]), "k": rng.choice([1, 5, 10])}
        if _cost(c) <= most:
            return c


# ----------------------------------------------------------------- the models

# the model file of each family: the published architecture with random weights
_WRITE = {"resnet34": (synth.write_resnet34, {}), "ecapa": (synth.write_ecapa, {}),
          "campplus": (synth.write_campplus, {}), "eres2net": (synth.write_eres2net, {}),
          "emotion": (synth.write_w2v2, {"kind": "emotion"})}
_files, _contexts, _weights = {}, {}, {}


def _model_file(model):
    if model not in _files:
        write, kw = _WRITE[model]
        _files[model] = os.path.join(tempfile.mkdtemp(prefix="cases_"), model + ".gguf")
        write(_files[model], 2024, **kw)
    return _files[model]


def _context(model):
    """The loaded model: one handle per process, as a server keeps it."""
    if model not in _contexts:
        _contexts[model] = lib.Context(_model_file(model))
    return _contexts[model]


def _model_weights(model):
    if model not in _weights:
        g = gguf.GGUFFile(_model_file(model))
        _weights[model] = (g.kv, {n: torch.from_numpy(np.array(g.array(n))).double().to(DEV) for n in g.tensors})
    return _weights[model]


# ----------------------------------------------------------------- the inputs

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _speech(seed, batch, n):
    """[batch][n] f32: voiced harmonics with a moving pitch, a syllable rhythm and background noise."""
    g = _gen(seed)
    u = torch.rand(batch, 4, generator=g, device=DEV, dtype=torch.float64)
    t = torch.arange(n, device=DEV, dtype=torch.float64)[None, :] / SR
    f0, vib, rate, depth = 90 + 160 * u[:, :1], 2 + 4 * u[:, 1:2], 2 + 4 * u[:, 2:3], 0.3 + 0.6 * u[:, 3:4]
    phase = 2 * math.pi * (f0 * t - 0.03 * f0 / vib / (2 * math.pi) * torch.cos(2 * math.pi * vib * t))
    x = torch.zeros(batch, n, device=DEV, dtype=torch.float64)
    for h in range(1, 13):
        x += torch.sin(h * phase) / h
    x *= 0.15 * (1 - depth * (0.5 + 0.5 * torch.cos(2 * math.pi * rate * t)))
    x += 0.004 * torch.randn(batch, n, generator=g, device=DEV, dtype=torch.float64)
    return x.float().contiguous()


def _normal(g, shape, std=1.0):
    return torch.randn(shape, generator=g, device=DEV) * std


def _frames(n):
    return 1 + (n - WIN) // HOP


def _w2v2_frames(n):
    for k, s in zip(synth.W2V2_BASE["conv_kernels"], synth.W2V2_BASE["conv_strides"]):
        n = (n - k) // s + 1
    return n


def _conv_inputs(case, seed):
    """The conv layer's inputs as a residual encoder meets them: post-ReLU maps, scaled weights."""
    g = _gen(seed)
    B, H, W, IC, OC, s = (case[k] for k in ("batch", "H", "W", "IC", "OC", "stride"))
    Ho, Wo = (H - 1) // s + 1, (W - 1) // s + 1
    x = _normal(g, (B, H, W, IC)).relu().half()
    w = _normal(g, (OC, 3, 3, IC), math.sqrt(2.0 / (9 * IC))).half()
    b = _normal(g, (OC,), 0.1)
    res = _normal(g, (B, Ho, Wo, OC)).relu().half() if s == 1 else None
    return x, w, b, res


def _asp_inputs(case, seed):
    g = _gen(seed)
    B, T, C = case["batch"], case["T"], case["C"]
    a1 = torch.tanh(_normal(g, (B, T, 128))).half()
    w = _normal(g, (C, 128), math.sqrt(2.0 / 128)).half()
    b = _normal(g, (C,), 0.01)
    x = (_normal(g, (B, T, C)).relu() * 1.2 - 0.1).half()
    return a1, w, b, x


def _identify_inputs(case, seed):
    """Unit rows; every second query is a noisy copy of an enrolled one, the others are strangers."""
    g = _gen(seed)
    B, N, D = case["batch"], case["rows"], case["dim"]
    reg = F.normalize(_normal(g, (N, D)), dim=1)
    at = torch.randint(0, N, (B,), generator=g, device=DEV)
    noise = F.normalize(_normal(g, (B, D)), dim=1)
    known = (torch.arange(B, device=DEV) % 2 == 0)[:, None]
    return F.normalize(torch.where(known, reg[at] + 0.6 * noise, noise), dim=1).contiguous(), reg.contiguous()


def _qkv(case, seed):
    return _normal(_gen(seed), (case["batch"], case["T"], 3 * 64 * case["heads"])).half()


# -------------------------------------------------------------------- prepare

def prepare(case, seed):
    L, kind = lib.lib(), case["kind"]
    st = {"case": case, "L": L}
    if kind in ("embed", "analyze"):
        ctx = _context(case["model"])
        st["ctx"] = ctx
        ctx.L.voicedetect_gpu_stream(ctx.ctx)       # the device is initialised and the weights are there
        st["pcm"] = _speech(seed, case["batch"], case["samples"])
        width = ctx.dim if kind == "embed" else ctx.analyze_outputs()
        st["out"] = torch.empty(case["batch"], width, device=DEV)
    elif kind == "fbank":
        B, n = case["batch"], case["samples"]
        cfg = lib.fbank_cfg()
        st["cfg"], st["pcm"] = cfg, _speech(seed, B, n)
        st["tables"] = torch.empty(L.vdk_fbank_tables_size(cfg), dtype=torch.uint8, device=DEV)
        lib.check(L.vdk_fbank_tables_fill(cfg, st["tables"].data_ptr()))
        st["work"] = torch.empty(L.vdk_fbank_workspace_size(cfg, B, n), dtype=torch.uint8, device=DEV)
        st["feats"] = torch.empty(B, MELS, _frames(n), device=DEV)
        st["mean"] = torch.empty(B, MELS, device=DEV)
    elif kind == "conv":
        x, w, b, res = _conv_inputs(case, seed)
        s, OC, IC = case["stride"], case["OC"], case["IC"]
        d = lib.ConvDesc()
        d.x, d.batch, d.H, d.W, d.IC = x.data_ptr(), case["batch"], case["H"], case["W"], IC
        d.w, d.OC, d.KH, d.KW = w.data_ptr(), OC, 3, 3
        d.stride_h = d.stride_w = s
        d.pad_h = d.pad_w = d.dil_h = d.dil_w = 1
        # the chunk-major copy of the weights that a loaded model keeps beside them
        wc = w.view(OC, 9, IC // 16, 16).permute(2, 1, 0, 3).contiguous()
        d.w_chunked, d.bias, d.act, d.tile = wc.data_ptr(), b.data_ptr(), lib.ACT_RELU, -1
        if res is not None:
            d.residual = res.data_ptr()
        y = torch.empty(case["batch"], (case["H"] - 1) // s + 1, (case["W"] - 1) // s + 1, OC, dtype=torch.half,
                        device=DEV)
        d.y = y.data_ptr()
        st.update(d=d, y=y, keep=(x, w, b, res, wc))
    elif kind == "attention":
        st["qkv"] = _qkv(case, seed)
        st["out"] = torch.empty(case["batch"], case["T"], 64 * case["heads"], dtype=torch.half, device=DEV)
    elif kind == "asp":
        st["in"] = _asp_inputs(case, seed)
        st["out"] = torch.empty(case["batch"], 2 * case["C"], device=DEV)
    else:
        B, N, k = case["batch"], case["rows"], case["k"]
        st["q"], st["reg"] = _identify_inputs(case, seed)
        st["work"] = torch.empty(L.vdk_registry_topk_workspace_size(B, N, k), dtype=torch.uint8, device=DEV)
        st["idx"] = torch.empty(B, k, dtype=torch.int32, device=DEV)
        st["score"] = torch.empty(B, k, device=DEV)
    torch.cuda.synchronize()
    return st


# ------------------------------------------------------------------------ run

def run(st):
    L, case = st["L"], st["case"]
    kind = case["kind"]
    if kind == "embed":
        st["ctx"].embed_device_async(st["pcm"].data_ptr(), case["batch"], case["samples"], st["out"].data_ptr())
        return st["out"]
    if kind == "analyze":
        st["ctx"].analyze_device_async(st["pcm"].data_ptr(), case["batch"], case["samples"], st["out"].data_ptr())
        return st["out"]
    if kind == "fbank":
        lib.check(L.vdk_fbank_ex(st["cfg"], st["tables"].data_ptr(), st["pcm"].data_ptr(), case["batch"],
                                 case["samples"], st["feats"].data_ptr(), st["mean"].data_ptr(),
                                 st["work"].data_ptr(), st["work"].numel(), None))
        return st["feats"], st["mean"]
    if kind == "conv":
        lib.check(L.vdk_conv2d_ex(st["d"], None))
        return st["y"]
    if kind == "attention":
        lib.check(L.vdk_attention(st["qkv"].data_ptr(), case["batch"], case["T"], case["heads"], 64, 0.125,
                                  st["out"].data_ptr(), None))
        return st["out"]
    if kind == "asp":
        a1, w, b, x = st["in"]
        C = case["C"]
        lib.check(L.vdk_asp_attn_pool(a1.data_ptr(), 128, w.data_ptr(), b.data_ptr(), 128, x.data_ptr(), C,
                                      case["batch"], case["T"], C, 1e-12, st["out"].data_ptr(), None))
        return st["out"]
    lib.check(L.vdk_registry_topk(st["q"].data_ptr(), case["batch"], st["reg"].data_ptr(), case["rows"],
                                  case["dim"], case["k"], st["work"].data_ptr(), st["work"].numel(),
                                  st["idx"].data_ptr(), st["score"].data_ptr(), None))
    return st["idx"], st["score"]


# ----------------------------------------------------------------------- work

def _resnet34_layers(T):
    """(multiply-adds, weights) of WeSpeaker ResNet34 on T frames."""
    H, W = MELS, T
    ma, nw = 9 * 32 * H * W, 9 * 32
    for ic, oc, s, down in synth.resnet34_spec():
        H, W = (H - 1) // s + 1, (W - 1) // s + 1
        for k in (9 * ic * oc, 9 * oc * oc, ic * oc if down else 0):
            ma, nw = ma + k * H * W, nw + k
    fc = 2 * 256 * H * 256
    return ma + fc, nw + fc


def _ecapa_layers(T):
    block = 2 * 1024 * 1024 + 7 * 3 * 128 * 128
    per = 5 * 80 * 1024 + 3 * block + 3072 * 1536 + 1536 * 128 + 128 * 1536
    once = 3 * 2 * 1024 * 128 + 3072 * 128 + 3072 * 192
    return per * T + once, per + once


def _campplus_layers(T):
    ma, nw, H, k = 9 * 32 * MELS * T, 9 * 32, MELS, 9 * 32 * 32
    for s in (2, 1, 2, 1):
        H //= s
        n = 2 * k + (32 * 32 if s == 2 else 0)
        ma, nw = ma + n * H * T, nw + n
    H //= 2
    ma, nw = ma + k * H * T, nw + k
    Tp, C = (T - 1) // 2 + 1, 128
    k = 5 * 32 * H * 128
    ma, nw = ma + k * Tp, nw + k
    for layers in (12, 24, 16):
        for _ in range(layers):
            k = C * 128 + 3 * 128 * 32
            ma, nw, C = ma + k * Tp, nw + k + 128 * 64 + 64 * 32, C + 32
        k, C = C * (C // 2), C // 2
        ma, nw = ma + k * Tp, nw + k
    return ma + 2 * C * 192, nw + 2 * C * 192


def _eres2net_layers(T):
    H, W, ma, nw, ic = MELS, T, 9 * 32 * MELS * T, 9 * 32, 32
    for li, (blocks, stride) in enumerate(zip((3, 4, 6, 3), (1, 2, 2, 2))):
        planes = 32 << li
        width = planes // 2
        for bi in range(blocks):
            s = stride if bi == 0 else 1
            H, W = (H - 1) // s + 1, (W - 1) // s + 1
            k = ic * 2 * width + 2 * 9 * width * width + 2 * width * 2 * planes
            k += 2 * width * (width // 4) + (width // 4) * width if li >= 2 else 0
            k += ic * 2 * planes if s != 1 or ic != 2 * planes else 0
            ma, nw, ic = ma + k * H * W, nw + k, 2 * planes
        if li >= 1:
            k = 9 * planes * 2 * planes + 4 * planes * (planes // 2) + (planes // 2) * 2 * planes
            ma, nw = ma + k * H * W, nw + k
    fc = 2 * 512 * H * 512
    return ma + fc, nw + fc


def _emotion_layers(n):
    ma, nw, ic = 0, 0, 1
    for k, s in zip(synth.W2V2_BASE["conv_kernels"], synth.W2V2_BASE["conv_strides"]):
        n = (n - k) // s + 1
        ma, nw, ic = ma + k * ic * 512 * n, nw + k * ic * 512, 512
    per = 512 * 768 + 768 * 48 * 128 + 12 * (4 * 768 * 768 + 2 * 768 * 3072) + 768 * 256
    return ma + per * n + 12 * 2 * 768 * n * n, nw + per


_LAYERS = {"resnet34": _resnet34_layers, "ecapa": _ecapa_layers, "campplus": _campplus_layers,
           "eres2net": _eres2net_layers}
_EMB = {"resnet34": 256, "ecapa": 192, "campplus": 192, "eres2net": 512}


def work(case):
    kind, B = case["kind"], case["batch"]
    if kind == "embed":
        ma, nw = _LAYERS[case["model"]](_frames(case["samples"]))
        return {"bytes": 4 * B * (case["samples"] + _EMB[case["model"]]) + 2 * nw, "flops": 2 * B * ma}
    if kind == "analyze":
        ma, nw = _emotion_layers(case["samples"])
        return {"bytes": 4 * B * (case["samples"] + 4) + 2 * nw, "flops": 2 * B * ma}
    if kind == "fbank":
        T = _frames(case["samples"])
        # a real 512-point transform, the power spectrum and the mel filters of each frame
        return {"bytes": 4 * B * (case["samples"] + MELS * T + MELS),
                "flops": B * T * (2.5 * NFFT * 9 + 3 * 257 + 4 * 257)}
    if kind == "conv":
        s, IC, OC = case["stride"], case["IC"], case["OC"]
        out = ((case["H"] - 1) // s + 1) * ((case["W"] - 1) // s + 1)
        return {"bytes": 2 * (B * case["H"] * case["W"] * IC + 9 * IC * OC + B * out * OC * (2 if s == 1 else 1)),
                "flops": 2 * 9 * IC * OC * B * out}
    if kind == "attention":
        T, H = case["T"], 64 * case["heads"]
        return {"bytes": 2 * B * T * 4 * H, "flops": 4 * B * T * T * H}
    if kind == "asp":
        T, C = case["T"], case["C"]
        return {"bytes": 2 * B * T * (C + 128) + 2 * 128 * C + 8 * B * C, "flops": 2 * B * T * C * (128 + 4)}
    return {"bytes": 4 * (B + case["rows"]) * case["dim"] + 8 * B * case["k"],
            "flops": 2 * B * case["rows"] * case["dim"]}


def _cost(case):
    w = work(case)
    return max(w["bytes"], w["flops"] / 50)


# ------------------------------------------------------------------ tolerance

def tolerance(case):
    """About four times what each path was measured to differ from exact()."""
    kind = case["kind"]
    if kind == "embed":
        # f16 activations and weights through 30 to 100 layers (measured 2e-4, 2.4e-4, 9e-4); ERes2Net in split-f16 (6e-5)
        return {"rel": {"resnet34": 1e-3, "ecapa": 1e-3, "campplus": 4e-3, "eres2net": 3e-4}[case["model"]]}
    if kind == "analyze":
        return {"rel": 1.2e-3}                  # f16 operands through 7 convs and 12 transformer layers (3e-4)
    if kind == "fbank":
        return {"rel": 2e-6, "max": 5e-5}       # f32 framing and results of a 64-bit transform (4e-7)
    if kind == "conv":
        return {"rel": 1e-3, "max": 4e-3}       # f16 store of an f32 sum (2e-4)
    if kind == "attention":
        return {"rel": 1.2e-3, "max": 1e-2}     # f16 probabilities and store (3e-4)
    if kind == "asp":
        return {"rel": 1e-6, "max": 1e-5}       # f32 logits, 64-bit sums (3e-8)
    return {"rel": 1e-7, "differ": 0.0}         # 64-bit sums rounded to f32 (3e-8), whole indexes


# ---------------------------------------------------------------------- exact

def _conv2d(x, w, b=None, stride=(1, 1), pad=(0, 0), dil=(1, 1)):
    """x [C][H][W], w [OC][C][KH][KW], f64, as one matrix product of its columns."""
    oc, ic, kh, kw = w.shape
    Ho = (x.shape[1] + 2 * pad[0] - dil[0] * (kh - 1) - 1) // stride[0] + 1
    Wo = (x.shape[2] + 2 * pad[1] - dil[1] * (kw - 1) - 1) // stride[1] + 1
    cols = F.unfold(x[None], (kh, kw), dilation=dil, padding=pad, stride=stride)[0]
    y = (w.reshape(oc, -1) @ cols).view(oc, Ho, Wo)
    return y if b is None else y + b[:, None, None]


def _conv1d(x, w, b=None, stride=1, pad=0, dil=1, reflect=False):
    """x [C][T], w [OC][C][K] (or [OC][C])."""
    w = w[:, :, None] if w.dim() == 2 else w
    if reflect and pad:
        x, pad = F.pad(x[None], (pad, pad), mode="reflect")[0], 0
    return _conv2d(x[:, None], w[:, :, None], b, (1, stride), (0, pad), (1, dil))[:, 0]


def _log_mel(pcm):
    """[n] -> Kaldi log-mel [MELS][T] without the mean subtraction."""
    dev = pcm.device
    x = pcm.double().unfold(0, WIN, HOP)
    x = x - x.mean(1, keepdim=True)
    pre = float(np.float32(0.97))
    x = x - pre * torch.cat([x[:, :1], x[:, :-1]], 1)
    i = torch.arange(WIN, device=dev, dtype=torch.float64)
    x = x * (0.5 - 0.5 * torch.cos(2 * math.pi * i / (WIN - 1))) ** 0.85
    p = torch.fft.rfft(x, NFFT).abs() ** 2
    mel = lambda f: 1127.0 * np.log(1.0 + f / 700.0)  # noqa: E731
    lo, hi = mel(20.0), mel(SR / 2)
    edge = lo + np.arange(MELS + 2) * (hi - lo) / (MELS + 1)
    m = mel(np.arange(NFFT // 2 + 1) * SR / NFFT)[None, :]
    left, mid, right = edge[:-2, None], edge[1:-1, None], edge[2:, None]
    fb = np.where((m > left) & (m <= mid), (m - left) / (mid - left),
                  np.where((m > mid) & (m < right), (right - m) / (right - mid), 0.0))
    e = p @ torch.from_numpy(fb).to(dev).T
    return torch.log(e.clamp_min(float(np.finfo(np.float32).eps))).T.contiguous()


def _features(pcm):
    f = _log_mel(pcm)
    return f - f.mean(1, keepdim=True)


def _tstp(x, eps):
    """[C][H][W] -> [mean ; std] over time, unbiased variance."""
    return torch.cat([x.mean(2).reshape(-1), (x.var(2, unbiased=True) + eps).sqrt().reshape(-1)])


def _unit(v):
    return v / v.norm()


def _exact_resnet34(kv, W, pcm):
    g = lambda name: kv["voicedetect.resnet." + name]  # noqa: E731
    x = _conv2d(_features(pcm)[None], W[g("stem_weight")], W[g("stem_bias")], pad=(1, 1)).relu()
    for i, s in enumerate(g("stride")):
        h = _conv2d(x, W[g("conv1_weight")[i]], W[g("conv1_bias")[i]], (s, s), (1, 1)).relu()
        down = g("down_weight")[i]
        sc = _conv2d(x, W[down], W[g("down_bias")[i]], (s, s)) if down else x
        x = (_conv2d(h, W[g("conv2_weight")[i]], W[g("conv2_bias")[i]], pad=(1, 1)) + sc).relu()
    return _unit(W[g("seg_weight")] @ _tstp(x, 1e-8) + W[g("seg_bias")])


def _bn(W, p, x, eps=1e-5):
    k = W[p + ".weight"] / (W[p + ".running_var"] + eps).sqrt()
    b = W[p + ".bias"] - k * W[p + ".running_mean"]
    return x * k[:, None] + b[:, None] if x.dim() == 2 else x * k + b


def _exact_ecapa(kv, W, pcm):
    def tdnn(x, p, dil=1):
        w = W[p + ".conv.conv.weight"]
        pad = (w.shape[2] - 1) // 2 * dil if w.dim() == 3 else 0
        return _bn(W, p + ".norm.norm", _conv1d(x, w, W[p + ".conv.conv.bias"], 1, pad, dil, True).relu())

    x, outs = tdnn(_features(pcm), "blocks.0"), []
    for i in (1, 2, 3):
        p = "blocks.%d" % i
        xs = tdnn(x, p + ".tdnn1").chunk(8)
        ys = [xs[0]]
        for j in range(1, 8):
            ys.append(tdnn(xs[j] if j == 1 else xs[j] + ys[-1], "%s.res2net_block.blocks.%d" % (p, j - 1), i + 1))
        y = tdnn(torch.cat(ys), p + ".tdnn2")
        se = lambda v, n: _conv1d(v, W[p + ".se_block.conv%d.conv.weight" % n],  # noqa: E731
                                  W[p + ".se_block.conv%d.conv.bias" % n])
        x = y * torch.sigmoid(se(se(y.mean(1, keepdim=True), 1).relu(), 2)) + x
        outs.append(x)
    x = tdnn(torch.cat(outs), "mfa")
    m, sd = x.mean(1, keepdim=True), x.var(1, unbiased=False, keepdim=True).clamp_min(1e-12).sqrt()
    a = torch.tanh(tdnn(torch.cat([x, m.expand_as(x), sd.expand_as(x)]), "asp.tdnn"))
    a = torch.softmax(_conv1d(a, W["asp.conv.conv.weight"], W["asp.conv.conv.bias"]), 1)
    mu = (a * x).sum(1)
    sd = (a * (x - mu[:, None]) ** 2).sum(1).clamp_min(1e-12).sqrt()
    p = _bn(W, "asp_bn.norm", torch.cat([mu, sd]))
    return _unit(_conv1d(p[:, None], W["fc.conv.weight"], W["fc.conv.bias"])[:, 0])


def _exact_campplus(kv, W, pcm):
    names = zip(kv["voicedetect.campplus.conv_weight"], kv["voicedetect.campplus.conv_bias"])
    layers = iter([(W[w], W[b] if b else None) for w, b in names])
    bns = iter(kv["voicedetect.campplus.bn_prefix"])
    x = _conv2d(_features(pcm)[None], *next(layers), pad=(1, 1)).relu()
    for s in (2, 1, 2, 1):
        h = _conv2d(x, *next(layers), stride=(s, 1), pad=(1, 1)).relu()
        c2 = next(layers)
        sc = _conv2d(x, *next(layers), stride=(s, 1)) if s == 2 else x
        x = (_conv2d(h, *c2, pad=(1, 1)) + sc).relu()
    x = _conv2d(x, *next(layers), stride=(2, 1), pad=(1, 1)).relu()
    h = _conv1d(x.reshape(-1, x.shape[2]), *next(layers), stride=2, pad=2).relu()
    T = h.shape[1]
    for bi, (n, dil) in enumerate(zip((12, 24, 16), (1, 2, 2))):
        for _ in range(n):
            c = _conv1d(_bn(W, next(bns), h).relu(), *next(layers)).relu()
            y = _conv1d(c, *next(layers), pad=dil, dil=dil)
            seg = torch.cat([s.sum(1, keepdim=True).expand_as(s) / 100 for s in c.split(100, 1)], 1)
            ctx = c.mean(1, keepdim=True) + seg
            z = _conv1d(_conv1d(ctx, *next(layers)).relu(), *next(layers))
            h = torch.cat([h, y * torch.sigmoid(z)])
        h = _conv1d(_bn(W, next(bns), h).relu(), *next(layers))
        h = h.relu() if bi == 2 else h
    e = _conv1d(_tstp(h[:, None], 0.0)[:, None], *next(layers))[:, 0]
    var, mean = (W[kv["voicedetect.campplus.emb_bn_" + k]] for k in ("var", "mean"))
    return _unit((e - mean) / (var + 1e-5).sqrt())


def _exact_eres2net(kv, W, pcm):
    g = lambda name: kv["voicedetect.eres2net." + name]  # noqa: E731
    layers = iter(zip(g("conv_weight"), g("conv_bias"), g("conv_stride")))

    def conv(x):
        w, b, s = next(layers)
        w = W[w] if W[w].dim() == 4 else W[w][:, :, None, None]
        return _conv2d(x, w, W[b] if b else None, (s, s), ((w.shape[2] - 1) // 2,) * 2)

    def aff(x, ds):
        z = torch.tanh(conv(F.silu(conv(torch.cat([x, ds])))))
        return (x + ds) + z * (x - ds)

    def layer(x, planes, n, stride, fuse):
        for i in range(n):
            s = stride if i == 0 else 1
            a, b = conv(x).clamp(0, 20).chunk(2)
            y0 = conv(a).clamp(0, 20)
            y1 = conv(aff(y0, b) if fuse else y0 + b).clamp(0, 20)
            y = conv(torch.cat([y0, y1]))
            sc = conv(x) if s != 1 or x.shape[0] != 2 * planes else x
            x = (y + sc).clamp(0, 20)
        return x

    x = conv(_features(pcm)[None]).relu()
    o1 = layer(x, 32, 3, 1, False)
    o2 = layer(o1, 64, 4, 2, False)
    fused = aff(o2, conv(o1))
    o3 = layer(o2, 128, 6, 2, True)
    fused = aff(o3, conv(fused))
    o4 = layer(o3, 256, 3, 2, True)
    fused = aff(o4, conv(fused))
    return _unit(W[g("seg_weight")] @ _tstp(fused, 1e-8) + W[g("seg_bias")])


def _exact_emotion(kv, W, pcm):
    gelu = lambda v: 0.5 * v * (1 + torch.erf(v / math.sqrt(2.0)))  # noqa: E731
    lin = lambda v, p: v @ W[p + ".weight"].T + W[p + ".bias"]      # noqa: E731

    def ln(v, p):
        v = v - v.mean(-1, keepdim=True)
        return v / ((v * v).mean(-1, keepdim=True) + 1e-5).sqrt() * W[p + ".weight"] + W[p + ".bias"]

    h = pcm.double()[None]
    for i, s in enumerate(synth.W2V2_BASE["conv_strides"]):
        p = "w2v2.feature_extractor.conv_layers.%d" % i
        h = _conv1d(h, W[p + ".conv.weight"], None, s)
        if i == 0:
            h = (h - h.mean(1, keepdim=True)) / (h.var(1, unbiased=False, keepdim=True) + 1e-5).sqrt()
            h = h * W[p + ".layer_norm.weight"][:, None] + W[p + ".layer_norm.bias"][:, None]
        h = gelu(h)
    h = lin(ln(h.T, "w2v2.feature_projection.layer_norm"), "w2v2.feature_projection.projection")
    T, H = h.shape
    p = "w2v2.encoder.pos_conv_embed.conv"
    v = W[p + ".weight_v"]
    w = v * (W[p + ".weight_g"].reshape(-1) / (v * v).sum((0, 1)).sqrt())
    c = H // 16
    pos = torch.cat([_conv1d(h.T[i * c:(i + 1) * c].contiguous(), w[i * c:(i + 1) * c], None, 1, 64)
                     for i in range(16)])
    h = ln(h + gelu(pos[:, :-1] + W[p + ".bias"][:, None]).T, "w2v2.encoder.layer_norm")
    weights = torch.softmax(W["layer_weights"].reshape(-1), 0)
    total = weights[0] * h
    for i in range(12):
        p = "w2v2.encoder.layers.%d" % i
        heads = [lin(h, "%s.attention.%s_proj" % (p, n)) for n in "qkv"]
        o = []
        for j in range(0, H, 64):
            q, k, v = (t[:, j:j + 64] for t in heads)
            o.append(torch.softmax(q @ k.T / 8.0, 1) @ v)
        h = ln(h + lin(torch.cat(o, 1), p + ".attention.out_proj"), p + ".layer_norm")
        f = lin(gelu(lin(h, p + ".feed_forward.intermediate_dense")), p + ".feed_forward.output_dense")
        h = ln(h + f, p + ".final_layer_norm")
        total = total + weights[i + 1] * h
    return lin(lin(total, "projector").mean(0), "classifier")


_EXACT = {"resnet34": _exact_resnet34, "ecapa": _exact_ecapa, "campplus": _exact_campplus,
          "eres2net": _exact_eres2net, "emotion": _exact_emotion}


def exact(case, seed):
    kind, B = case["kind"], case["batch"]
    if kind in ("embed", "analyze"):
        kv, W = _model_weights(case["model"])
        pcm = _speech(seed, B, case["samples"])
        return torch.stack([_EXACT[case["model"]](kv, W, pcm[i]) for i in range(B)])
    if kind == "fbank":
        f = torch.stack([_log_mel(x) for x in _speech(seed, B, case["samples"])])
        return f, f.mean(2)
    if kind == "conv":
        x, w, b, res = _conv_inputs(case, seed)
        w, b, s = w.double().permute(0, 3, 1, 2).contiguous(), b.double(), case["stride"]
        out = []
        for i in range(B):
            y = _conv2d(x[i].double().permute(2, 0, 1).contiguous(), w, b, (s, s), (1, 1)).permute(1, 2, 0)
            out.append((y if res is None else y + res[i].double()).relu().float())
        return torch.stack(out)
    if kind == "attention":
        H, out = 64 * case["heads"], []
        for x in _qkv(case, seed):
            q, k, v = x.double().split(H, 1)
            out.append(torch.cat([torch.softmax(q[:, j:j + 64] @ k[:, j:j + 64].T * 0.125, 1) @ v[:, j:j + 64]
                                  for j in range(0, H, 64)], 1))
        return torch.stack(out)
    if kind == "asp":
        a1, w, b, x = _asp_inputs(case, seed)
        out = []
        for i in range(B):
            xi = x[i].double()
            a = torch.softmax(a1[i].double() @ w.double().T + b.double(), 0)
            mu = (a * xi).sum(0)
            out.append(torch.cat([mu, (a * (xi - mu) ** 2).sum(0).clamp_min(1e-12).sqrt()]))
        return torch.stack(out)
    q, reg = _identify_inputs(case, seed)
    score, idx = (q.double() @ reg.double().T).topk(case["k"], 1)
    return idx, score
