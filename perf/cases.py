"""Performance cases of the int8 inference path: what a program built on this package
asks of it, over the sizes such programs use.

Eight kinds of work, each through the package's public entry points and on data that is
already on the device:

  mlp        a small dynamically quantized MLP, driven from Python: host time and launches count
  dynamic    one dynamically quantized Linear (``quantize_dynamic``), from one row to a whole batch
  token      a Linear with per-token activation scales and float16 output, as a language model runs
             it: a few rows while decoding, thousands in prefill
  wonly      group-wise weight-only int4 / int8 products on float32 activations
  roundtrip  calibration and conversion of a tensor: range -> qparams -> quantize -> dequantize,
             or fake-quantize in their place
  resnet     a statically quantized ResNet-50 replayed from a graph
  vit        a dynamically quantized ViT-B/16 replayed from a graph
  lstm       a dynamically quantized LSTM over a batch of sequences

``listed()`` gives named cases, ``draw(rng)`` one more of the same ranges; ``prepare`` makes the
inputs and what a program keeps between calls, ``run`` is one pass.
"""

from __future__ import annotations

import functools

import numpy as np
import torch

import lucid_amd as L
import lucid_amd.nn as nn
import lucid_amd.nn.functional as F
import lucid_amd.nn.intrinsic as nni
import lucid_amd.nn.quantized as nnq
import lucid_amd.nn.quantized.dynamic as nnqd
import lucid_amd.quantization as Q
from lucid_amd import _C, _ops
from lucid_amd.quantization import _qgemm

_LARGEST_GEMM = 2048 * 4096 * 11008


def listed():
    return [
        # the MNIST-sized classifier of the benchmark: a batch of 64 costs less than issuing it
        dict(name="mlp_784_256_10_b64", kind="mlp", batch=64, sizes="784,256,10"),
        # one token through the wide Linear of a 7B-parameter decoder's MLP: bound by reading the weight
        dict(name="dynamic_m1", kind="dynamic", m=1, k=4096, n=11008, bias=True),
        # a Linear whose sizes suit no tile: 333 rows of 1000 features onto 1001 outputs
        dict(name="dynamic_m333_ragged", kind="dynamic", m=333, k=1000, n=1001, bias=True),
        # sixteen sequences decoded together, per-token scales
        dict(name="token_m16", kind="token", m=16, k=4096, n=11008),
        # a prefill of 2048 tokens, the quantization of its activations included
        dict(name="token_m2048", kind="token", m=2048, k=4096, n=11008),
        # 4-bit weight-only decoding of one sequence
        dict(name="wonly4_m1", kind="wonly", m=1, k=4096, n=11008, bits=4, group=64),
        # 8-bit weight-only decoding of sixteen sequences
        dict(name="wonly8_m16", kind="wonly", m=16, k=4096, n=11008, bits=8, group=64),
        # a 4-bit weight-only prompt of 333 tokens
        dict(name="wonly4_m333", kind="wonly", m=333, k=4096, n=11008, bits=4, group=128),
        # a checkpoint-sized tensor: per-channel range, qparams, codes and back
        dict(name="roundtrip_4096x4096x16", kind="roundtrip", a=4096, b=4096, c=16, axis=0, symmetric=True,
             unsigned=False, fake=False),
        # image classification at the benchmark's batch sizes
        dict(name="resnet50_b32", kind="resnet", batch=32, size=224, parts=2),
        dict(name="vit_b16_b64", kind="vit", batch=64),
        # two recurrent layers over 64 steps of 16 sequences
        dict(name="lstm_512x2_t64_b16", kind="lstm", inputs=512, hidden=512, layers=2, steps=64, batch=16,
             bidirectional=False, batch_first=False),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def _features(rng, lo, hi):
    """A feature count: mostly a multiple of 16, one time in four any number."""
    v = _log_int(rng, lo, hi)
    return v if rng.random() < 0.25 else max(16, v // 16 * 16)


def draw(rng):
    kind = rng.choice(["mlp", "dynamic", "token", "wonly", "roundtrip", "resnet", "vit", "lstm"])
    if kind == "mlp":
        return dict(kind=kind, batch=_log_int(rng, 1, 256),
                    sizes=f"{_features(rng, 32, 1024)},{_features(rng, 32, 512)},{_log_int(rng, 2, 64)}")
    if kind in ("dynamic", "token"):
        while True:
            m, k, n = _log_int(rng, 1, 2048), _features(rng, 128, 8192), _log_int(rng, 64, 11008)
            if m * k * n <= _LARGEST_GEMM:
                break
        return dict(kind=kind, m=m, k=k, n=n, **({"bias": rng.random() < 0.5} if kind == "dynamic" else {}))
    if kind == "wonly":
        group = rng.choice([32, 64, 128])
        while True:
            m, k, n = _log_int(rng, 1, 1024), group * _log_int(rng, 4, 8192 // group), _log_int(rng, 256, 11008)
            if m * k * n <= 1024 * 4096 * 4096:
                break
        return dict(kind=kind, m=m, k=k, n=n, bits=rng.choice([4, 8]), group=group)
    if kind == "roundtrip":
        while True:
            a, b, c = _log_int(rng, 1, 8192), _log_int(rng, 16, 8192), _log_int(rng, 1, 64)
            if 10_000 <= a * b * c <= 1 << 28:
                break
        return dict(kind=kind, a=a, b=b, c=c, axis=rng.choice([-1, 0, 1, 2]), symmetric=rng.random() < 0.5,
                    unsigned=rng.random() < 0.5, fake=rng.random() < 0.3)
    if kind == "resnet":
        batch = _log_int(rng, 1, 32)
        return dict(kind=kind, batch=batch, size=rng.randint(96, 224), parts=min(batch, rng.choice([1, 2])))
    if kind == "vit":
        return dict(kind=kind, batch=_log_int(rng, 1, 64))
    return dict(kind=kind, inputs=_features(rng, 32, 512), hidden=_features(rng, 32, 512), layers=rng.choice([1, 2]),
                steps=_log_int(rng, 4, 64), batch=_log_int(rng, 1, 64), bidirectional=rng.random() < 0.3,
                batch_first=rng.random() < 0.5)


# ---------------------------------------------------------------- tensors
class _Memory:
    """A package tensor's device memory as torch sees it; keeps the tensor alive."""

    def __init__(self, t):
        self.t = t
        self.__cuda_array_interface__ = {"shape": t.shape, "typestr": np.dtype(t.dtype.np).str, "strides": None,
                                         "data": (t.data_ptr, False), "version": 2}


def _out(t):
    return torch.as_tensor(_Memory(t), device="cuda")


def _in(v):
    """A torch device tensor as a package tensor of its own."""
    t = L.Tensor.empty(tuple(v.shape), str(v.dtype).removeprefix("torch."), "hip")
    _out(t).copy_(v)
    return t


def _normal(gen, *shape, std=1.0):
    return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32) * std


def _linear(gen, k, n, bias=True):
    """A float Linear with the weight spread of a trained one."""
    lin = nn.Linear(k, n, bias=bias)
    lin.register_buffer("weight", _in(_normal(gen, n, k, std=0.02)))
    if bias:
        lin.register_buffer("bias", _in(_normal(gen, n, std=0.02)))
    return lin


# ---------------------------------------------------------------- the two networks
def _calibrated(mod, lo, hi):
    """``mod`` with the observer state of a calibration that saw the range [lo, hi]."""
    mod.qconfig = Q.get_default_qconfig()
    obs = mod.activation_post_process = Q.MinMaxObserver()
    obs.register_buffer("min_val", L.tensor(np.float32(lo), device="hip"))
    obs.register_buffer("max_val", L.tensor(np.float32(hi), device="hip"))
    return mod


def _qconv(gen, cin, cout, k, stride=1, relu=True, gain=2 ** 0.5):
    conv = nn.Conv2d(cin, cout, k, stride=stride, padding=k // 2)
    conv.register_buffer("weight", _in(_normal(gen, cout, cin, k, k, std=gain / (cin * k * k) ** 0.5)))
    conv.register_buffer("bias", _in(_normal(gen, cout, std=0.02)))
    if relu:
        return nnq.ConvReLU2d.from_float(_calibrated(nni.ConvReLU2d(conv, nn.ReLU()), 0.0, 6.0))
    return nnq.Conv2d.from_float(_calibrated(conv, -4.0, 4.0))


class _Bottleneck(nn.Module):
    def __init__(self, gen, cin, planes, stride):
        super().__init__()
        self.conv1 = _qconv(gen, cin, planes, 1)
        self.conv2 = _qconv(gen, planes, planes, 3, stride)
        self.conv3 = _qconv(gen, planes, 4 * planes, 1, relu=False, gain=0.5)
        self.down = _qconv(gen, cin, 4 * planes, 1, stride, relu=False, gain=1.0) if cin != 4 * planes else None
        self.join = nnq.QFunctional.from_float(_calibrated(nnq.FloatFunctional(), 0.0, 8.0))

    def forward(self, x):
        identity = x if self.down is None else self.down(x)
        return self.conv3(self.conv2(self.conv1(x)), join=(identity, self.join, True))


_STAGES = ((64, 3, 1), (128, 4, 2), (256, 6, 2), (512, 3, 2))  # planes, blocks, stride of the first


class _ResNet50(nn.Module):
    """Statically quantized, float32 images in, float32 logits out."""

    def __init__(self, gen):
        super().__init__()
        self.quant = nnq.Quantize.from_float(_calibrated(nnq.QuantStub(), 0.0, 1.0))
        self.conv1, self.pool = _qconv(gen, 3, 64, 7, 2), nn.MaxPool2d(3, 2, 1)
        cin, blocks = 64, []
        for planes, count, stride in _STAGES:
            for i in range(count):
                blocks.append(_Bottleneck(gen, cin, planes, stride if i == 0 else 1))
                cin = 4 * planes
        self.blocks, self.avg, self.flatten = nn.Sequential(*blocks), nn.AdaptiveAvgPool2d(1), nn.Flatten()
        fc = _linear(gen, cin, 1000)
        self.fc, self.dequant = nnq.Linear.from_float(_calibrated(fc, -4.0, 4.0)), nnq.DeQuantize()

    def forward(self, x):
        x = self.blocks(self.pool(self.conv1(x, quantize=self.quant)))
        return self.dequant(self.fc(self.flatten(self.avg(x))))


def _resnet50_macs(size):
    """Multiply-accumulates of one image."""
    out = lambda n, k, s: (n + 2 * (k // 2) - k) // s + 1
    h = out(size, 7, 2)
    macs, h, cin = h * h * 64 * 3 * 49, out(h, 3, 2), 64
    for planes, count, stride in _STAGES:
        for i in range(count):
            o = out(h, 3, stride) if i == 0 else h
            macs += h * h * cin * planes + o * o * planes * planes * 9 + o * o * planes * 4 * planes
            if cin != 4 * planes:
                macs += o * o * cin * 4 * planes
            h, cin = o, 4 * planes
    return macs + cin * 1000


_DIM, _HEADS, _HIDDEN, _DEPTH, _TOKENS, _PATCH = 768, 12, 3072, 12, 197, 16


class _EncoderBlock(nn.Module):
    def __init__(self, gen):
        super().__init__()
        self.norm1, self.norm2 = _layer_norm(gen), _layer_norm(gen)
        self.qkv, self.proj = _linear(gen, _DIM, 3 * _DIM), _linear(gen, _DIM, _DIM)
        self.fc1, self.fc2 = _linear(gen, _DIM, _HIDDEN), _linear(gen, _HIDDEN, _DIM)

    @staticmethod
    def _normed(norm, lin, x, **kw):
        q, scale, zp = F.layer_norm_dynamic_quantize(x, norm.normalized_shape, norm.weight, norm.bias, norm.eps,
                                                     lin.act_qdtype)
        return lin.forward_quantized(q, scale, zp, x.shape[:-1], **kw)

    def forward(self, x):
        a = F.scaled_dot_product_attention_qkv(self._normed(self.norm1, self.qkv, x), _HEADS, track_range=True)
        x = self.proj(a, residual=x)
        return self.fc2(self._normed(self.norm2, self.fc1, x, activation="gelu", track_range=True), residual=x)


def _layer_norm(gen, track_range=True):
    ln = nn.LayerNorm(_DIM, eps=1e-6, track_range=track_range)
    ln.register_buffer("weight", _in(1 + _normal(gen, _DIM, std=0.02)))
    ln.register_buffer("bias", _in(_normal(gen, _DIM, std=0.02)))
    return ln


class _ViT(nn.Module):
    """ViT-B/16 with dynamically quantized Linears, float32 images in, float32 logits out."""

    def __init__(self, gen):
        super().__init__()
        for name, shape in (("patch_weight", (_DIM, 3 * _PATCH ** 2)), ("patch_bias", (_DIM,)), ("cls", (_DIM,)),
                            ("pos", (_TOKENS, _DIM))):
            self.register_buffer(name, _in(_normal(gen, *shape, std=0.02)))
        self.blocks = nn.Sequential(*[_EncoderBlock(gen) for _ in range(_DEPTH)])
        self.norm, self.head = _layer_norm(gen, track_range=False), _linear(gen, _DIM, 1000)
        Q.quantize_dynamic(self, inplace=True)

    def forward(self, x):
        b, c, h, w = x.shape
        tokens, cls = L.Tensor.empty((b, _TOKENS, _DIM)), L.Tensor.empty((b, _DIM))
        _C.call("lq_patch_embed_f32", x.data_ptr, self.patch_weight.data_ptr, self.patch_bias.data_ptr,
                self.cls.data_ptr, self.pos.data_ptr, tokens.data_ptr, b, c, h, w, _PATCH, _DIM, None)
        tokens = self.norm(self.blocks(tokens))
        _C.call("lq_gather_rows_f32", tokens.data_ptr, _TOKENS * _DIM, cls.data_ptr, b, _DIM, None)
        return self.head(cls)


@functools.lru_cache(maxsize=None)
def _model(kind):
    """A deployed network: its weights are the same for every batch."""
    gen = torch.Generator(device="cuda").manual_seed(1)
    return (_ResNet50 if kind == "resnet" else _ViT)(gen)


# ---------------------------------------------------------------- a case's state and one pass over it
def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind, s = case["kind"], dict(case)
    if kind == "mlp":
        k, h, n = (int(v) for v in case["sizes"].split(","))
        s["model"] = Q.quantize_dynamic(nn.Sequential(_linear(gen, k, h), nn.ReLU(), _linear(gen, h, n)))
        s["x"] = _in(_normal(gen, case["batch"], k))
    elif kind == "dynamic":
        s["model"] = nnqd.Linear.from_float(_linear(gen, case["k"], case["n"], case["bias"]))
        s["x"] = _in(_normal(gen, case["m"], case["k"]))
    elif kind == "token":
        w = _in(_normal(gen, case["n"], case["k"], std=0.02))
        scale, zp = Q.calculate_qparams(*Q.minmax(w, ch_axis=0), Q.per_channel_symmetric, Q.qint8)
        s["w"], s["scale"] = Q.quantize(w, scale, zp, Q.qint8, ch_axis=0), scale
        s["bias"] = _in(_normal(gen, case["n"], std=0.02).half())
        s["x"] = _in(_normal(gen, case["m"], case["k"]))
    elif kind == "wonly":
        w = _in(_normal(gen, case["n"], case["k"], std=0.02))
        s["w"] = _qgemm.quantize(w, case["group"], case["bits"])
        s["x"] = _in(_normal(gen, case["m"], case["k"]))
    elif kind == "roundtrip":
        x = _normal(gen, case["a"], case["b"], case["c"])
        x[torch.rand(x.shape, generator=gen, device="cuda") < 1e-3] *= 20  # the outliers of real activations
        s["x"] = _in(x)
    elif kind in ("resnet", "vit"):
        size = case.get("size", 224)
        x = _in(torch.rand((case["batch"], 3, size, size), generator=gen, device="cuda"))
        s["x"], s["model"], parts = x, _model(kind), case.get("parts", 1)
        if parts > 1:
            for i in range(parts):
                s["model"](x.row_range(case["batch"] * i // parts, case["batch"] * (i + 1) // parts))
            s["graph"] = L.graph.capture_split(s["model"], x, parts)
            s["y"] = _out(s["graph"].output)
        else:
            s["model"](x)
            with L.graph.capture() as s["graph"]:
                y = s["model"](x)
            s["y"] = _out(y)
    elif kind == "lstm":
        lstm = nn.LSTM(case["inputs"], case["hidden"], num_layers=case["layers"], batch_first=case["batch_first"],
                       bidirectional=case["bidirectional"])
        s["model"] = nnqd.LSTM.from_float(lstm)
        lead = (case["batch"], case["steps"]) if case["batch_first"] else (case["steps"], case["batch"])
        s["x"] = _in(_normal(gen, *lead, case["inputs"]))
    return s


def run(s):
    kind = s["kind"]
    if kind in ("mlp", "dynamic"):
        return _out(s["model"](s["x"]))
    if kind == "token":
        xq, scale, _ = Q.quantize_rows_dynamic(s["x"], Q.per_channel_symmetric, Q.qint8)
        return _out(_ops.qlinear_i8(xq, s["w"], a_scale=scale, w_scale=s["scale"], bias=s["bias"],
                                    out_mode=_ops.OUT_F16))
    if kind == "wonly":
        return _out(_qgemm.quantized_matmul(s["x"], *s["w"], group_size=s["group"], bits=s["bits"]))
    if kind == "roundtrip":
        axis, qd = None if s["axis"] < 0 else s["axis"], Q.quint8 if s["unsigned"] else Q.qint8
        scheme = {(True, True): Q.per_tensor_symmetric, (True, False): Q.per_tensor_affine,
                  (False, True): Q.per_channel_symmetric, (False, False): Q.per_channel_affine}[axis is None, s["symmetric"]]
        scale, zp = Q.calculate_qparams(*Q.minmax(s["x"], ch_axis=axis), scheme, qd)
        if s["fake"]:
            y = Q.fake_quantize(s["x"], scale, zp, qd.quant_min, qd.quant_max, ch_axis=axis)
            return _out(scale), _out(zp), _out(y)
        q = Q.quantize(s["x"], scale, zp, qd, ch_axis=axis)
        return _out(scale), _out(zp), _out(q), _out(Q.dequantize(q, scale, zp, ch_axis=axis))
    if kind in ("resnet", "vit"):
        s["graph"].replay()
        return s["y"]
    y, (h, c) = s["model"](s["x"])
    return _out(y), _out(h), _out(c)


# ---------------------------------------------------------------- what a pass cannot do without
def work(case):
    kind = case["kind"]
    if kind == "mlp":
        k, h, n = (int(v) for v in case["sizes"].split(","))
        b = case["batch"]
        return {"bytes": 4 * b * (k + n) + h * (k + n) + 12 * (h + n), "flops": 2 * b * h * (k + n)}
    if kind in ("dynamic", "token"):
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": 4 * m * k + n * k + 8 * n + m * n * (4 if kind == "dynamic" else 2), "flops": 2 * m * k * n}
    if kind == "wonly":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": 4 * m * (k + n) + n * k * case["bits"] // 8 + 8 * n * k // case["group"], "flops": 2 * m * k * n}
    if kind == "roundtrip":
        count = case["a"] * case["b"] * case["c"]
        return {"bytes": count * (8 if case["fake"] else 10 if case["unsigned"] else 9), "flops": 0}
    if kind == "resnet":
        return {"bytes": 25.5e6 + case["batch"] * (12 * case["size"] ** 2 + 4000),
                "flops": 2 * case["batch"] * _resnet50_macs(case["size"])}
    if kind == "vit":
        linears = _DEPTH * _TOKENS * _DIM * (4 * _DIM + 2 * _HIDDEN) + _DIM * 1000
        attention, patch = _DEPTH * 2 * _TOKENS ** 2 * _DIM, (_TOKENS - 1) * _DIM * 3 * _PATCH ** 2
        return {"bytes": 88e6 + case["batch"] * (12 * 224 ** 2 + 4000),
                "flops": 2 * case["batch"] * (linears + attention + patch)}
    dirs, hid, rows = 2 if case["bidirectional"] else 1, case["hidden"], case["steps"] * case["batch"]
    weights, fan = 0, case["inputs"]
    for _ in range(case["layers"]):
        weights, fan = weights + dirs * 4 * hid * (fan + hid), dirs * hid
    return {"bytes": weights + 4 * rows * (case["inputs"] + fan), "flops": 2 * rows * weights}


def tolerance(case):
    """What another correct implementation may differ by: four times the distance of the path to
    itself evaluated in float64 (``vit``: to itself on images one float32 rounding apart)."""
    kind = case["kind"]
    if kind in ("roundtrip", "resnet"):
        return "exact"  # integer codes and the float values they stand for: every step is defined to the bit
    if kind in ("mlp", "dynamic"):
        return {"rel": 2.5e-4, "max": 0.016}  # an activation on a rounding tie lands on the next code
    if kind == "token":
        return {"rel": 8e-4, "max": 2e-3}  # one rounding to float16
    if kind == "vit":
        return {"rel": 0.03, "max": 0.35}  # twelve layers of ties: two evaluations drift by whole codes
    return {"rel": 4e-6, "max": 4e-5} if kind == "wonly" else {"rel": 1.5e-6, "max": 1.3e-5}
