"""Dynamic-quantized ``Linear`` on the hip int8 GEMM.

Mirrors ``lucid/nn/quantized/dynamic/linear.py:64-124``: buffers
``weight_int8`` / ``weight_scale`` / ``weight_zero_point`` / ``bias``,
attribute ``act_qdtype = quint8``, ``from_float(mod, dtype=qint8)``.  Per
forward: global min / max of the input -> affine qparams -> activation codes
-> int8 GEMM -> float32 output (not requantized).  All four steps are device
kernels; the activation zero point is read by the GEMM from device memory, so
the forward never waits for the host.
"""

from __future__ import annotations

import ctypes as C

import numpy as np

from .... import _C, _ops
from .... import _tensor as T
from .... import graph as _graph
from ...._tensor import Tensor
from ....quantization._functional import minmax, quantize
from ....quantization._qparams import calculate_qparams
from ....quantization._qscheme import QDtype, per_channel_symmetric, per_tensor_affine, qint8, quint8
from ...module import Module
from .._utils import forget_weight_zero_points, storage_offset, weight_zero_points


# Rows of activation codes that fit the LDS of the one-launch kernel of small layers: wider layers
# quantize in a launch of their own, whatever the batch.
SMALL_LINEAR_MAX_K = 6080


def _one_launch_pays(M: int, K: int, N: int) -> bool:
    """Whether the one-launch kernel of a small layer beats quantizing (4 us) and multiplying (5 us and
    up) in two.  Its blocks each take the range of all of x and quantize 16 rows: about 4 us + 0.043 us per
    1000 activations + 2.4 us per 1000 of K, one round of 256 blocks.  Measured: 64 x 784 -> 256 8.0 us,
    7 x 1024 -> 1024 7.2, 16 x 4096 -> 1024 16.5, 32 x 2048 -> 4096 (512 blocks) 22.7, 16 x 4096 -> 11008 48.5."""
    return (1 < M <= 64 and 0 < K <= SMALL_LINEAR_MAX_K and M * K <= 65536
            and ((M + 15) // 16) * ((N + 15) // 16) <= 256 and 43 * M * K + 2400 * K <= 6_000_000)


# Bytes of activation codes that the one-call route keeps in the stream's scratch at most (from there on the
# launches it saves are about 1 % of a layer's time).
MAX_CODE_BYTES = 1 << 28


def _code_row_bytes(K: int) -> int:
    """Length of a row of codes, of the weight or the activation, as the one-call route lays it out."""
    return K if K % 16 == 0 else (K + 63) // 64 * 64


def _one_call_takes(M: int, K: int) -> bool:
    """Whether ``lq_dynamic_linear_f32`` takes M rows of K: the padded row within the int32 accumulator, the padded
    codes within the scratch they may have (a short ragged row grows to 64 bytes)."""
    ld = _code_row_bytes(K)
    return ld <= 131071 and M * ld <= MAX_CODE_BYTES


def _kernel_operands(lin, N: int, K: int):
    """Weight, scales and bias of ``lin`` if they are what the one-call kernels read by address, else ``None``.  A
    loaded state may hold other types or sizes, or a weight that is an unaligned view: the separate operators take
    those, or refuse them.  (Straight from the registry, and once: these calls are bound by what they cost the host.)"""
    b, f32, n = lin._buffers, T.float32, (N,)
    w, scale, bias = taken = b["weight_int8"], b["weight_scale"], b["bias"]
    if (w.dtype is T.int8 and w.shape == (N, K) and not w._offset & 15 and scale.dtype is f32 and scale.shape == n
            and (bias is None or bias.dtype is f32 and bias.shape == n)):
        return taken
    return None


def _keep(*derived) -> None:
    """Keeps ``(layer, name, value)``, derived from the weights by work that this call has issued, for the calls to come:
    once that work is done, since those may run on other streams.  (Waited for behind the call's own launches: before
    them it made a first call 25 to 45 us longer.)  A capture only records the work: it is then part of every
    replay, and nothing is kept."""
    capturing = C.c_int()
    _C.check(_C.load().lq_stream_is_capturing(C.byref(capturing), _C.current_stream()))
    if capturing.value or _graph.is_capturing():
        return
    _C.call("lq_sync", None)
    for lin, name, value in derived:
        setattr(lin, name, value)


# What the one launch for two layers holds: the first layer's row of codes, the hidden row of the block that runs the second.
PAIR_MAX_K, PAIR_MAX_HIDDEN = 1024, 511


def _pair_in_one_launch(M: int, K1: int, N1: int, N2: int) -> bool:
    """Whether ``lq_dynamic_mlp2_rows_f32`` takes the pair: what its blocks (all of x) and the last one of them (all of
    the hidden activation) keep in registers."""
    return (M > 0 and 0 < K1 <= PAIR_MAX_K and 0 < N1 <= PAIR_MAX_HIDDEN and 0 < N2 <= 64 and M * K1 <= 65536
            and (M <= 64 or M * _code_row_bytes(N1) <= 32768 and (M + 15) // 16 * ((N1 + 15) // 16) <= 192))


def fused_pair(first, relu_between: bool, second, x):
    """``second(relu(first(x)))`` (or without the ReLU) for two dynamic ``Linear`` layers on a small
    activation as ONE launch (``lq_dynamic_mlp2_small_f32``: the last block of layer 1 to finish
    reduces the hidden activation's min / max and runs layer 2; ``lq_dynamic_mlp2_small_rows_f32`` where a weight's
    rows are no whole 16 bytes or the hidden layer is wide; ``lq_dynamic_mlp2_rows_f32`` for more than 64 rows), beyond
    it as two calls with the ReLU in the first one's epilogue, or ``None`` when the shapes or operands do not qualify.
    Same bits as calling the modules one after the other.  Per forward, ReLU between: 91-32-58 of 12 rows in one launch 12.6
    us (32 in three calls, which is what their host side takes), 64 rows of 784-496-10 17.9 (33), 148 of 32-48-15 14.0, 256
    of 256-128-64 18.1, 2048 of 32-16-8 24.9 (28.5 in two calls)."""
    if not (isinstance(first, Linear) and isinstance(second, Linear) and isinstance(x, Tensor)):
        return None
    if x.device != "hip" or x.dtype != T.float32 or x._grid is not None or x._range is not None:
        return None
    K1, N1, N2 = first.in_features, first.out_features, second.out_features
    if x.ndim < 1 or x.shape[-1] != K1 or second.in_features != N1:
        return None
    M = x.numel // K1 if K1 else 0
    small = _pair_in_one_launch(M, K1, N1, N2)
    rows = small and (M > 64 or K1 % 16 != 0 or N1 % 16 != 0 or N1 > 256)
    if rows and x.data_ptr % 16:
        small = False
    if not small and not relu_between:
        return None
    if first.act_qdtype is not second.act_qdtype:
        return None
    if weight_zero_points(first) is not None or weight_zero_points(second) is not None:
        return None
    if not small:
        h = first._one_call(x, M, K1, N1, 1) if M else None
        return None if h is None else second(h)
    taken1, taken2 = _kernel_operands(first, N1, K1), _kernel_operands(second, N2, N1)
    if taken1 is None or taken2 is None:
        return None
    (w1, scale1, bias1), (w2, scale2, bias2) = taken1, taken2
    wsum1, wsum2 = first._wsum, second._wsum
    fresh = ()
    if wsum1 is None or wsum2 is None:
        wsum1, wsum2 = first._weight_sums(), second._weight_sums()
        fresh = ((first, "_wsum", wsum1), (second, "_wsum", wsum2))
    qd = first.act_qdtype
    y = Tensor.empty((*x.shape[:-1], N2), T.float32, "hip")
    b1, b2 = None if bias1 is None else bias1.data_ptr, None if bias2 is None else bias2.data_ptr
    grid = (0, qd.quant_min, qd.quant_max, int(qd.signed), 1e-8, storage_offset(qd))
    if rows:
        padded = []
        for lin, w, K in ((first, w1, K1), (second, w2, N1)):
            rows = (w, K) if K % 16 == 0 else lin._wrows
            if rows is None:
                rows = lin._weight_rows()
                fresh += ((lin, "_wrows", rows),)
            padded.append(rows)
        (w1, ld1), (w2, ld2) = padded
        _C.call("lq_dynamic_mlp2_small_rows_f32" if M <= 64 else "lq_dynamic_mlp2_rows_f32", x.data_ptr, M, K1, w1.data_ptr,
                ld1, N1, scale1.data_ptr, wsum1.data_ptr, b1, int(relu_between), w2.data_ptr, ld2, N2, scale2.data_ptr,
                wsum2.data_ptr, b2, 0, *grid, y.data_ptr, None)
    else:
        _C.call("lq_dynamic_mlp2_small_f32", x.data_ptr, M, K1, w1.data_ptr, N1, scale1.data_ptr, wsum1.data_ptr,
                b1, int(relu_between), w2.data_ptr, N2, scale2.data_ptr, wsum2.data_ptr, b2, 0, *grid, y.data_ptr, None)
    if fresh:
        _keep(*fresh)
    return y


class Linear(Module):
    def __init__(self, in_features: int, out_features: int, bias: bool = True) -> None:
        super().__init__()
        self.in_features = in_features
        self.out_features = out_features
        self.weight_ch_axis = 0
        self.act_qdtype: QDtype = quint8
        self.register_buffer("weight_int8", T.tensor(
            np.zeros((out_features, in_features), np.int8), device="hip"))
        self.register_buffer("weight_scale", T.tensor(np.ones(out_features, np.float32), device="hip"))
        self.register_buffer("weight_zero_point", T.tensor(
            np.zeros(out_features, np.float32), device="hip"))
        self.register_buffer("bias", T.tensor(np.zeros(out_features, np.float32), device="hip")
                             if bias else None)
        self._wsum = None
        self._wrows = None

    # (a buffer that is assigned is another weight as much as one that is loaded)
    def register_buffer(self, name: str, tensor: Tensor | None) -> None:
        super().register_buffer(name, tensor)
        self._state_loaded(name)

    def __setattr__(self, name, value) -> None:
        super().__setattr__(name, value)
        self._state_loaded(name)

    def _state_loaded(self, name: str) -> None:
        if name == "weight_int8":
            self._wsum = self._wrows = None
        if name == "weight_zero_point":
            forget_weight_zero_points(self)

    def _weight_sums(self) -> Tensor:
        """The sums of the weight's rows."""
        return _ops.rowsum_i8(self._buffers["weight_int8"])

    def _weight_rows(self) -> tuple[Tensor, int]:
        """The weight codes of a ragged layer in rows of a multiple of 64 bytes with zeros behind them, and that length."""
        N, K = self.out_features, self.in_features
        ld = _code_row_bytes(K)
        rows = Tensor.empty((N, ld), T.int8, "hip")
        _C.call("lq_fill_bytes", rows.data_ptr, 0, rows.nbytes, None)
        _C.call("lq_d2d_rows", rows.data_ptr, ld, self._buffers["weight_int8"].data_ptr, K, K, N, None)
        return rows, ld

    def _one_call(self, x: Tensor, M: int, K: int, N: int, relu: int) -> Tensor | None:
        """min / max, qparams, codes, GEMM, bias and an optional ReLU behind one call (the same bits as the separate
        operators), or ``None`` where that call does not take the layer."""
        if (weight_zero_points(self) is not None or not _one_call_takes(M, K)
                or (taken := _kernel_operands(self, N, K)) is None):
            return None
        w, scale, bias = taken
        wsum, fresh = self._wsum, ()
        if wsum is None:
            wsum = self._weight_sums()
            fresh = ((self, "_wsum", wsum),)
        qd = self.act_qdtype
        y = Tensor.empty((*x.shape[:-1], N), T.float32, "hip")
        grid = (relu, 0, qd.quant_min, qd.quant_max, int(qd.signed), 1e-8, storage_offset(qd))
        b = None if bias is None else bias.data_ptr
        at, ldw = x.data_ptr if M else None, K
        if K % 16:
            if self._wrows is not None:
                w, ldw = self._wrows
            else:
                w, ldw = rows = self._weight_rows()
                fresh += ((self, "_wrows", rows),)
        if 1 < M <= 64 and _one_launch_pays(M, K, N) and (ldw == K or at % 16 == 0):
            if ldw == K:
                _C.call("lq_dynamic_linear_small_f32", at, M, K, w.data_ptr, N, scale.data_ptr, wsum.data_ptr, b, *grid,
                        y.data_ptr, None)
            else:
                _C.call("lq_dynamic_linear_small_rows_f32", at, M, K, w.data_ptr, ldw, N, scale.data_ptr, wsum.data_ptr, b,
                        *grid, y.data_ptr, None)
        else:
            _C.call("lq_dynamic_linear_f32", at, M, K, w.data_ptr, ldw, N, scale.data_ptr, wsum.data_ptr, b, *grid,
                    y.data_ptr if M else None, None)
        if fresh:
            _keep(*fresh)
        return y

    def forward(self, x: Tensor, residual: Tensor | None = None, activation: str | None = None,
                track_range: bool = False) -> Tensor:
        """Beyond Lucid's signature, all inside the GEMM epilogue: ``residual`` is added to
        the output (``x_res + linear(x)`` in one kernel); ``activation="gelu"`` applies the
        exact-erf GELU to it (``gelu(linear(x))``); ``track_range`` keeps the min / max of
        what is written, for the next dynamic-quantized layer."""
        if activation not in (None, "gelu"):
            raise ValueError(f"dynamic.Linear: unknown fused activation {activation!r}")
        if not isinstance(x, Tensor) or x.device != "hip":
            raise _C.DeviceMismatch("dynamic.Linear: input must be a tensor on the 'hip' device")
        if x.dtype != T.float32:
            raise _C.DtypeMismatch(f"dynamic.Linear expects float32 input, got {x.dtype}")
        K, N = self.in_features, self.out_features
        if x.shape[-1] != K:
            raise _C.ShapeMismatch(f"expected last dim {K}, got {x.shape}")
        M = x.numel // K
        if x._range is None and residual is None and activation is None and not track_range:
            y = self._one_call(x, M, K, N, 0)
            if y is not None:
                return y
        qd = self.act_qdtype
        off = storage_offset(qd)
        xq = Tensor.empty((M, K), T.int8, "hip")
        small = x._range is None and x.numel <= (1 << 18)
        if small:
            # min / max, qparams and codes of a small activation in one launch (same bits)
            x_scale = Tensor.empty((), T.float32, "hip")
            x_zp = Tensor.empty((), T.float32, "hip")
            _C.call("lq_quantize_tensor_dynamic_i8", x.data_ptr if x.numel else None, x.numel, 0, qd.quant_min,
                    qd.quant_max, int(qd.signed), 1e-8, off, x_scale.data_ptr, x_zp.data_ptr, None, None,
                    xq.data_ptr if x.numel else None, None)
        elif x._range is not None:
            # the kernel that wrote x kept its min / max: qparams and codes straight from them
            x_scale = Tensor.empty((), T.float32, "hip")
            x_zp = Tensor.empty((), T.float32, "hip")
            _C.call("lq_quantize_from_range_i8", x.data_ptr if x.numel else None, x.numel, x._range.data_ptr, 0, qd.quant_min,
                    qd.quant_max, int(qd.signed), 1e-8, off, x_scale.data_ptr, x_zp.data_ptr,
                    xq.data_ptr if x.numel else None, None)
        else:
            mn, mx = minmax(x)
            x_scale, x_zp = calculate_qparams(mn, mx, per_tensor_affine, qd)
            _C.call("lq_quantize", x.data_ptr, xq.data_ptr, _C.I8, off, 1, 1, x.numel,
                    x_scale.data_ptr, x_zp.data_ptr, 0, qd.quant_min, qd.quant_max, None)
        return self.forward_quantized(xq, x_scale, x_zp, x.shape[:-1], residual, activation, track_range)

    def forward_quantized(self, xq: Tensor, x_scale: Tensor, x_zp: Tensor, lead_shape, residual: Tensor | None = None,
                          activation: str | None = None, track_range: bool = False) -> Tensor:
        """The layer on an activation that is already quantized with this layer's activation
        grid (``act_qdtype``, per-tensor affine, device-side ``x_scale`` / ``x_zp``): what
        ``forward`` does after its own quantization, for a producer that writes codes directly
        (``functional.layer_norm_dynamic_quantize``)."""
        N = self.out_features
        off = storage_offset(self.act_qdtype)
        kept = self._wsum
        wsum = self._weight_sums() if kept is None else kept
        rng = None
        w_zp = weight_zero_points(self)
        if track_range and w_zp is not None:
            raise NotImplementedError("dynamic.Linear: track_range (an extension of this backend) is "
                                      "not available with affine weights")
        if track_range:
            from ...functional import _new_range
            rng = _new_range()
        y = _ops.qlinear_i8(xq, self.weight_int8, a_zp=off, a_zp_dev=x_zp, a_scale=x_scale,
                            w_scale=self.weight_scale, wsum=wsum, bias=self.bias,
                            out_mode=_ops.OUT_F32, residual=residual, gelu=activation == "gelu",
                            range_buf=rng, w_zp=w_zp)
        y = y.reshape(*lead_shape, N)
        y._range = rng
        if kept is None:
            _keep((self, "_wsum", wsum))
        return y

    @classmethod
    def from_float(cls, mod, dtype: QDtype = qint8) -> "Linear":
        """Quantize a float ``Linear``'s weight, no calibration
        (``dynamic/linear.py:101-120``)."""
        from ....quantization.observer import PerChannelMinMaxObserver

        qmod = cls(mod.in_features, mod.out_features, bias=mod.bias is not None)
        weight = mod.weight.to("hip")
        obs = PerChannelMinMaxObserver(ch_axis=0, qscheme=per_channel_symmetric, qdtype=dtype)
        obs(weight)
        scale, zero_point = obs.calculate_qparams()
        if dtype.storage != "int8":
            raise NotImplementedError(f"dynamic.Linear weights must use int8 storage, got {dtype!r}")
        qmod.register_buffer("weight_int8", quantize(weight, scale, zero_point, dtype, ch_axis=0))
        qmod.register_buffer("weight_scale", scale)
        qmod.register_buffer("weight_zero_point", zero_point)
        if mod.bias is not None:
            qmod.register_buffer("bias", mod.bias.to("hip"))
        return qmod

    def extra_repr(self) -> str:
        return f"in_features={self.in_features}, out_features={self.out_features}, dynamic=True"
