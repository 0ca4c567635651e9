"""4-bit linear layers with the class names, buffer names/shapes and forward semantics
of the reference's ``qlinear4bit/nn/linear.py``.  The forward is one fused launch
(GEMM + dequant + bias) instead of matmul + dequant + a torch add; ``fused = False`` on
a module switches back to the reference's three-step sequence (same bits).

Buffers (the state_dict contract): ``weight`` uint8 [N, K/2]; ``weight_scales`` [N, 1]
(``weight_scales_1/_2`` for the dual layers); ``weight_zeros*`` fp16 [N, 1] for the
asymmetric layers; optional ``bias`` [N].
"""
from __future__ import annotations

import contextlib
import functools
import threading

import torch

from .. import _HIP as _ops
from ..tools import quantization as quant_utils
from ..tools import tensor_utils
from ._calls import native_call
from .quantizer import AsymQuantizer, AsymQuantizer8bit, SymQuantizer  # noqa: F401  (re-exported like the reference)

_INT4_LEVELS = 2 ** 4


_making = threading.local()
_copying = threading.RLock()   # held where a layer's copy of its weight and the key it goes by are put in place


def _weight_key(layer):
    """What a copy of the layer's weight goes by: the copy is the weight's while this is what it was before it was made."""
    w = layer.weight
    return w._version, w.data_ptr(), w.device


def _put_copy(layer, name, key_name, make, wait):
    """Make the layer's copy of its weight (buffer ``name``) and the key it goes by.  Another stream may read the copy as soon
    as the key is there, and its user knows nothing of the launch that writes a copy made on the way in a forward: that one is
    waited for (``wait``), once per weight (a first 8-bit call of 8 rows, 4096 x 4096: 62 -> 90 us).  While a graph is
    recorded nothing is written yet: the recording gets a copy without a key, and calls outside of it make their own."""
    with _copying:
        key = _weight_key(layer)
        with torch.inference_mode(False):
            copy = make(layer.weight)
        if copy.device.type == "cuda":
            with torch.cuda.device(copy.device):
                if torch.cuda.is_current_stream_capturing():
                    key = None
                elif wait:
                    torch.cuda.current_stream().synchronize()
        layer.register_buffer(name, copy, persistent=False)
        setattr(layer, key_name, key)


def _placeholder_weight(shape, dtype):
    """What a layer holds until weights are put in: small random codes, as in the reference."""
    if getattr(_making, "unfilled", False):
        return torch.empty(shape, dtype=dtype)
    return torch.randint(1, 7, shape, dtype=dtype, requires_grad=False)


def _unfilled(cls, *args, device=None, **kwargs):
    """A layer (on ``device``) whose whole weight the caller writes: without the random codes (14 of the 15 ms that
    converting a 4096 x 4096 layer took were the host's random numbers)."""
    _making.unfilled = True
    try:
        with contextlib.nullcontext() if device is None else torch.device(device):
            return cls(*args, **kwargs)
    finally:
        _making.unfilled = False


_STAGE_BYTES = 16 << 20   # pieces of a copy: two pinned buffers of this size at most
_STAGE_FROM = 1 << 20     # below, the synchronous copies cost less than the way round


def _store(*pairs):
    """dst.copy_(src) of every pair.  Converted on the GPU into a layer on the host, the tensors go through pinned memory
    (torch's pool of it keeps the buffers), all copies in flight at once and one piece of 16 MB emptied while the next one
    arrives: 4096 x 4096 codes in 0.25 ms (0.16 of them the transfer), where one synchronous copy into pageable memory after the
    other takes 0.46 and 0.03 more for each small tensor."""
    staged = [(d, s) for d, s in pairs if s.is_cuda and not d.is_cuda and s.dtype == d.dtype and s.shape == d.shape and
              s.is_contiguous() and d.is_contiguous()]
    if sum(s.nbytes for _, s in staged) < _STAGE_FROM or len({s.device for _, s in staged}) != 1:
        staged = []
    kept = {id(d) for d, _ in staged}
    for d, s in pairs:
        if id(d) not in kept:
            d.copy_(s)
    if not staged:
        return
    pieces = [[]]   # groups of (host bytes, device bytes, offset in the pinned buffer)
    fill = 0
    for d, s in sorted(staged, key=lambda p: p[1].nbytes):
        d, s = d.view(-1).view(torch.uint8), s.view(-1).view(torch.uint8)
        at = 0
        while at < s.numel():
            if fill == _STAGE_BYTES:
                pieces.append([])
                fill = 0
            n = min(_STAGE_BYTES - fill, s.numel() - at)
            pieces[-1].append((d[at:at + n], s[at:at + n], fill))
            at, fill = at + n, min(-(-(fill + n) // 256) * 256, _STAGE_BYTES)
    most = _STAGE_BYTES if len(pieces) > 1 else fill
    with torch.cuda.device(staged[0][1].device):
        pins = [torch.empty(most, dtype=torch.uint8, device="cpu", pin_memory=True) for _ in pieces[:2]]
        arrived = [torch.cuda.Event() for _ in pins]
        for k in range(len(pieces) + 1):
            if k < len(pieces):
                for _, s, at in pieces[k]:
                    pins[k & 1][at:at + s.numel()].copy_(s, non_blocking=True)
                arrived[k & 1].record()
            if k:
                arrived[k - 1 & 1].synchronize()
                for d, _, at in pieces[k - 1]:
                    d.copy_(pins[k - 1 & 1][at:at + d.numel()])


_move_codes = None


def _is_move(fn):
    """Whether ``fn``, handed to ``_apply``, is what torch.nn.Module.to or .cuda hand there: told by its code, taken down from a
    module that is asked to move and does not."""
    global _move_codes
    if _move_codes is None:
        class Asked(torch.nn.Module):
            def _apply(self, fn, recurse=True):
                codes.add(getattr(fn, "__code__", None))
                return self

        codes = set()
        Asked().to("cpu")
        Asked().cuda()
        _move_codes = codes - {None}
    return getattr(fn, "__code__", None) in _move_codes


class _MovesTogether(torch.nn.Module):
    """A layer's move from the host to a GPU.  torch copies buffer after buffer out of pageable memory, which the runtime has
    to pin first; here they go through pinned memory (torch's pool of it, two pieces of 16 MB at most), all copies in flight
    at once and one piece filled while the other one leaves: a 4096 x 4096 layer 310 - 480 -> 260 us, its
    conversion with the move 800 -> 700."""

    def _apply(self, fn, recurse=True):
        here = [t for t in self._buffers.values() if type(t) is torch.Tensor and t.device.type == "cpu" and
                t.layout is torch.strided and t.is_contiguous() and t.numel()]
        if sum(t.nbytes for t in here) < _STAGE_FROM or not _is_move(fn):
            return super()._apply(fn, recurse)
        there = _fetch(here, fn)
        return super()._apply(lambda t: there[id(t)] if id(t) in there else fn(t), recurse)


def _fetch(tensors, move):
    """{id(t): move(t)} of the host tensors that ``move`` takes to a GPU as they are."""
    # (device="cpu", here and below: the caller may have set another default device)
    like = {dtype: move(torch.empty(0, dtype=dtype, device="cpu")) for dtype in {t.dtype for t in tensors}}
    tensors = [t for t in {id(t): t for t in tensors}.values() if like[t.dtype].is_cuda and like[t.dtype].dtype == t.dtype]
    if not tensors:
        return {}
    device = like[tensors[0].dtype].device
    there = {}
    with torch.cuda.device(device):
        if torch.cuda.is_current_stream_capturing():
            return {}
        size = min(_STAGE_BYTES, sum(-(-t.nbytes // 256) * 256 for t in tensors))
        pins = [torch.empty(size, dtype=torch.uint8, device="cpu", pin_memory=True)]
        left = [torch.cuda.Event(), torch.cuda.Event()]
        k = fill = 0
        for t in tensors:
            there[id(t)] = out = torch.empty(t.shape, dtype=t.dtype, device=device)
            src, dst = t.view(-1).view(torch.uint8), out.view(-1).view(torch.uint8)
            at = 0
            while at < src.numel():
                if fill == size:   # this piece is full: on to the other one, once what it held has left
                    left[k].record()
                    k, fill = k ^ 1, 0
                    if len(pins) == 1:
                        pins.append(torch.empty(size, dtype=torch.uint8, device="cpu", pin_memory=True))
                    left[k].synchronize()
                n = min(size - fill, src.numel() - at)
                pin = pins[k][fill:fill + n]
                pin.copy_(src[at:at + n])
                dst[at:at + n].copy_(pin, non_blocking=True)
                at, fill = at + n, min(-(-(fill + n) // 256) * 256, size)
        torch.cuda.current_stream().synchronize()
    return there


def _bias_pair(new, module):
    return () if module.bias is None else ((new.bias, module.bias.data),)


def _pack_given(w, codes_of, scales, split=0):
    """Packed codes rint(w / scale) of a symmetric layer's ``from_float``: one pass on the GPU where the weight allows it,
    else pack_i4 of ``codes_of()``; both refuse codes outside [-8, 7]."""
    scales = [s.to(w.device) for s in scales]
    if _ops.weight_takes_one_pass(w) and all(s.dtype is torch.float16 for s in scales):
        q, bad = _ops.weight_quant_sym(w, *(s.contiguous() for s in scales), split=split)
        assert not int(bad), "value outside the int4 range"
        return q
    return quant_utils.pack_i4(codes_of().to(torch.int8))


def _asym_params(w: torch.Tensor):
    """Per-row scale / zero / codes the way the reference's ``from_linear`` computes them:
    max and min are taken over |W| (linear.py:129-136)."""
    aw = w.abs()
    w_max = aw.amax(dim=-1, keepdim=True)
    w_min = aw.amin(dim=-1, keepdim=True)
    scale = (w_max - w_min) / (_INT4_LEVELS - 1)
    zeros = (-w_min / scale).round().to(torch.float16)
    codes = torch.clamp(torch.round(w / scale) + zeros, 0, _INT4_LEVELS - 1)
    return scale, zeros, codes


_FP6_MIN_TILES = 32  # the rule for smaller settings is written in csrc/duq_host.cpp too


class _Linear4bitBase(_MovesTogether):
    fused = True
    # 6-bit float matrix path (not in the reference): taken when the layer holds a weight shadow
    # (enable_fp6) and the input brings one, for more rows than the integer decode kernel takes (64 of up to 8192
    # elements, 48 of up to 12288, 32 beyond) and at least fp6_min_tiles output tiles of 64 x 256, or more than 256
    # rows and 5/8 of that (below, the integer kernels' smaller tiles and the decode kernels do better).  Rows that the layer
    # gets unquantized, up to 1024 of 1024 elements and more, which the integer kernels take in one library call: ten times as
    # many tiles, twenty below 2048 elements, eight from 8192 on (_fp6_pays).  A setting below the default asks for the 6-bit
    # float path where these rules have the integer kernels ahead, and is taken as it is in either case.
    # Eager steps of Linear4bitASQ, 6-bit float against integer, us: 160 x 4096 x 4096 25.4 / 11.8, 512 x 4096 x 8192
    # 25.0 / 21.6, 768 x 4096 x 8192 26.9 / 29.2, 384 x 8192 x 8192 32.7 / 32.0, 512 x 8192 x 8192 33.9 / 35.0, 248 x 19968 x 17264 106 / 114, 1024 x 16384 x 4096 64.9 /
    # 63.2, 512 x 1536 x 16384 25.3 / 19.0, 768 x 1536 x 16384 25.0 / 27.4
    fp6_min_tiles = _FP6_MIN_TILES
    # Device memory that a call of some thousand rows may take for itself to make both operands' 6-bit float shadows, where the layer
    # holds none and that is faster (0: none, the integer kernel runs; same bits).  A graph's memory holds what its recording took.
    prefill_room_bytes = _ops.ROOM_BYTES
    _shadow_key = None

    def _finish(self, y):
        return y if self.bias is None else y + self.bias

    # ---- decode: quantizer + GEMM + dequant in one call (ONE launch up to eight rows of binary16 activations and for some hundred short ones) ----
    # _decode_spec: (epilogue mode, ((argument of _HIP.FusedDecode, buffer name), ...)) of a layer class that has a
    # one-launch form; the weight comes first.
    _decode_spec = None
    _decode = None

    def __getstate__(self):
        """A copy or a saved file of the layer goes without its prepared call, which holds addresses of this process."""
        state = self.__dict__.copy()
        state.pop("_decode", None)
        return state

    def _decode_call(self):
        """The layer's prepared one-launch call (``_HIP.FusedDecode``), rebuilt when a buffer was replaced (moved,
        cast, reloaded into a new tensor) or given other memory (``.data``); None for a layer that has none or is not on
        a GPU."""
        d = self._decode
        b = self._buffers
        if d is not None and d.holds(b):
            return d
        spec = self._decode_spec
        if spec is None:
            return None
        names = spec[1] + (("bias", "bias"),)
        held = tuple((buf, b.get(buf)) for _, buf in names)
        if not held[0][1].is_cuda:
            return None
        d = self._decode = _ops.FusedDecode(spec[0], **{arg: t for (arg, _), (_, t) in zip(names, held)}).prepare_for(held)
        return d

    def _decode_forward(self, x, clip=1.0, qmax=6, checked=False):
        """y for binary16 rows ``x`` when the layer takes them in one library call (up to eight rows, and more
        short ones while their tiles are one round of workgroups: one launch, quantizer inside; the others up to 1024: quantizer
        launch + GEMM launch), else None."""
        if not self.fused:
            return None
        d = self._decode_call()
        if d is None:
            return None
        K = d.K
        if K % 64 or x.shape[-1] != K:
            return None
        M = x.numel() // K
        if d._one.get(M, -1) < 0 and not d.admits(M):
            return None
        if M > 64 and self._fp6_pays(M):  # large enough for the 6-bit float path, and the layer holds a shadow
            return None
        return d.run(x, M, clip, qmax, checked)

    def _take_deferred(self, x):
        """A PackedQuantizedTensor that SymQuantizer handed on unquantized: the result of the one-call path, or None
        after quantizing it now (with the 6-bit float shadow when this layer will take that path)."""
        d = self._decode
        if d is not None and d.native is not None and self.fused:   # everything in native code; None: not the plain case
            y = d.native.take(self._buffers, x)
            if y is not None:
                return y
        y = self._decode_forward(x.source(), x._clip, x._qmax, True)
        if y is None:
            src = x._src
            rows = src.numel() // src.shape[-1]
            x.materialize(shadow=bool(self.fused and src.shape[-1] % 128 == 0 and self._fp6_pays(rows)))
        return y

    def enable_fp6(self):
        """Build the E3M2 shadow of ``weight`` (3/4 byte per element next to the 1/2 byte of the packed
        nibbles; not part of the state_dict; rebuilt when ``weight`` changes) on the current stream.  Results are
        bit-identical; large inputs run 20-25 % faster.  Needs out_features % 16 == 0 and in_features % 128 == 0."""
        self._build_shadow(wait=False)
        return self

    def _build_shadow(self, wait):
        assert self.weight.is_cuda, "the shadow is built on the GPU: move the layer there first"
        assert not self.weight.is_inference(), "the weight was made in torch.inference_mode() and counts no versions: a change " \
            "of it could not be told; build or move the layer outside"
        assert self.out_features % 16 == 0 and self.in_features % 128 == 0, \
            "the 6-bit float path needs out_features % 16 == 0 and in_features % 128 == 0"
        _put_copy(self, "weight_shadow", "_shadow_key", tensor_utils.weight_shadow, wait)

    def _fp6_ready(self):
        if self._buffers.get("weight_shadow") is None or self.weight.is_inference():
            return False
        if self._shadow_stale():   # weights were loaded or moved since
            with _copying:
                if self._shadow_stale():
                    self._build_shadow(wait=True)
        return True

    def _shadow_stale(self):
        return self._shadow_key != _weight_key(self) or self.weight_shadow.device != self.weight.device

    def _fp6_wanted(self, rows):
        tiles = -(-rows // 64) * -(-self.out_features // 256)
        decode_rows = 64 if self.in_features <= 8192 else (48 if self.in_features <= 12288 else 32)
        return self._fp6_ready() and rows > decode_rows and \
            (tiles >= self.fp6_min_tiles or (rows > 256 and 8 * tiles >= 5 * self.fp6_min_tiles))

    def _fp6_pays(self, rows):
        """The same for rows that are not quantized yet."""
        K, least = self.in_features, self.fp6_min_tiles
        if rows <= 1024 <= K and least >= _FP6_MIN_TILES and \
                -(-rows // 64) * -(-self.out_features // 256) < (8 if K >= 8192 else 10 if K >= 2048 else 20) * least:
            return False
        return self._fp6_wanted(rows)

    def _use_shadow(self, x):
        """The input's shadow is used when the layer is ready for it and the problem is large enough, or
        when the input brings nothing else."""
        if x.shadow_x is None:
            return False
        if x.quantized_x is None:
            assert self._fp6_ready(), "the input holds only a 6-bit float shadow: call enable_fp6() on the layer"
            return True
        return self._fp6_wanted(x.shadow_x.numel() // x.shadow_x.shape[-1])

    def _own_quantizer_decode(self, x):
        """Layers with their own AsymQuantizer: a few contiguous binary16 rows on the GPU run quantizer + GEMM +
        dequant as one launch (the quantizer inside the GEMM kernel, same bits); None for anything else."""
        d = self._decode
        if d is not None and d.native is not None and self.fused:
            y = d.native.take_rows(self._buffers, x)
            if y is not None:
                return y
        if type(x) is not torch.Tensor or x.dtype is not torch.float16 or not x.is_cuda or not x.is_contiguous() or \
                x.data_ptr() % 16:
            return None
        return self._decode_forward(x)

    def _quantize(self, x):
        """Own quantizer of the asymmetric layers: shadow only when this call will take the 6-bit float path."""
        rows = x.numel() // x.shape[-1]
        return self.quantizer(x, shadow="only" if self._fp6_pays(rows) else False)


@native_call("sym_layer")
class Linear4bitSQ(_Linear4bitBase):
    """Symmetric 4-bit linear layer; takes a PackedQuantizedTensor (linear.py:24-78)."""

    def __init__(self, in_features, out_features, bias=False, dtype=torch.float16):
        super().__init__()
        self.in_features = in_features
        self.out_features = out_features
        self.register_buffer("weight_scales", torch.zeros((out_features, 1), requires_grad=False))
        self.register_buffer("weight", _placeholder_weight((out_features, in_features // 2), torch.uint8))
        if bias:
            self.register_buffer("bias", torch.zeros((out_features), dtype=dtype))
        else:
            self.bias = None

    _decode_spec = (_ops.EPI_SYM, (("w", "weight"), ("w_scale_1", "weight_scales")))

    def forward(self, x):
        assert type(x) == tensor_utils.PackedQuantizedTensor  # quantized input is required
        if x._src is not None:  # up to 1024 rows straight from SymQuantizer: quantizer and GEMM in one library call
            y = self._take_deferred(x)
            if y is not None:
                return y
        xq, scales_x = x.quantized_x, x.scales_x
        if self.fused and self._use_shadow(x):
            return tensor_utils.linear_forward_shadow(_ops.EPI_SYM, x.shadow_x, scales_x, None, self.weight_shadow,
                                                      self.weight_scales, bias=self.bias)
        if self.fused:
            return tensor_utils.linear_forward(_ops.EPI_SYM, xq, scales_x, None, self.weight, self.weight_scales,
                                               bias=self.bias,
                                               room_bytes=self.prefill_room_bytes)
        acc = tensor_utils.matmul(xq, self.weight)
        return self._finish(tensor_utils.sym_dequant(acc, scales_x, self.weight_scales))

    @staticmethod
    def from_float(module: torch.nn.Linear, weight_scales=None):
        """Quantize ``module.weight`` with the given per-row scales: round(W / s), no clamp
        (pack_i4 rejects values outside [-8, 7]) (linear.py:58-78)."""
        w = module.weight.data
        make = Linear4bitSQ if weight_scales is None else functools.partial(_unfilled, Linear4bitSQ)
        new = make(module.in_features, module.out_features, bias=module.bias is not None, dtype=w.dtype).to(w.dtype)
        if weight_scales is not None:
            assert weight_scales.shape == (module.out_features, 1), "weight_scales should have shape (out_features, 1)"
            q = _pack_given(w, lambda: (w / weight_scales.to(w.device)).round(), (weight_scales,))
            _store((new.weight, q), (new.weight_scales, weight_scales.to(w.dtype)), *_bias_pair(new, module))
        return new


@native_call("own_layer")
class Linear4bitASQ(_Linear4bitBase):
    """Asymmetric 4-bit linear layer with its own AsymQuantizer (linear.py:80-145)."""

    def __init__(self, in_features, out_features, bias=False, require_quantizer=True):
        super().__init__()
        self.in_features = in_features
        self.out_features = out_features
        self.require_quantizer = require_quantizer
        self.register_buffer("weight_scales", torch.zeros((out_features, 1), requires_grad=False, dtype=torch.float16))
        self.register_buffer("weight_zeros", torch.zeros((out_features, 1), requires_grad=False, dtype=torch.float16))
        self.register_buffer("weight", _placeholder_weight((out_features, in_features // 2), torch.uint8))
        if bias:
            self.register_buffer("bias", torch.zeros((out_features), dtype=torch.float16))
        else:
            self.bias = None
        if require_quantizer:
            self.quantizer = AsymQuantizer()

    _decode_spec = (_ops.EPI_ASYM, (("w", "weight"), ("w_scale_1", "weight_scales"), ("w_zeros_1", "weight_zeros")))

    def forward(self, x):
        if self.require_quantizer:
            y = self._own_quantizer_decode(x)
            if y is not None:
                return y
            x = self._quantize(x) if self.fused else self.quantizer(x)
        assert type(x) == tensor_utils.PackedQuantizedTensor, \
            "Input should be quantized tensor, or require_quantizer should be passed as initial argument"
        xq, scales_x, zeros_x = x.quantized_x, x.scales_x, x.zeros_x
        if self.fused and self._use_shadow(x):
            return tensor_utils.linear_forward_shadow(_ops.EPI_ASYM, x.shadow_x, scales_x, zeros_x, self.weight_shadow,
                                                      self.weight_scales, self.weight_zeros, bias=self.bias)
        if self.fused:
            return tensor_utils.linear_forward(_ops.EPI_ASYM, xq, scales_x, zeros_x, self.weight, self.weight_scales,
                                               self.weight_zeros, bias=self.bias,
                                               room_bytes=self.prefill_room_bytes)
        acc = tensor_utils.matmul(xq, self.weight)
        return self._finish(tensor_utils.asym_dequant(acc, scales_x, zeros_x, self.weight_scales, self.weight_zeros))

    @classmethod
    def from_linear(cls, module: torch.nn.Linear, require_quantizer: bool = True):
        new = _unfilled(cls, module.in_features, module.out_features, bias=module.bias is not None,
                        require_quantizer=require_quantizer)
        w = module.weight.data
        if _ops.weight_takes_one_pass(w):
            q, ((scale, zeros),) = _ops.weight_quant_asym(w)
        else:
            scale, zeros, codes = _asym_params(w)
            q = quant_utils.pack_i4(codes.to(torch.int8), sym=False)
        _store((new.weight, q), (new.weight_scales, scale.to(torch.float16)), (new.weight_zeros, zeros.to(torch.float16)),
               *_bias_pair(new, module))
        return new


@native_call("own_layer")
class Linear4bitASQRowSum(_Linear4bitBase):
    """Asymmetric 4-bit linear layer with the exact zero-point correction.  Not in the
    reference: its Linear4bitASQ stores unsigned codes that the signed GEMM misreads
    (README.md:31-32) and its epilogue subtracts the zero points from the accumulator
    (src/kernels/quant.cu:167-168).  Here codes and zero points are stored minus 8, the signed
    GEMM is exact for them, and the epilogue applies
        y = s_x * s_w * (acc - z_x * (R_w - K * z_w) - z_w * R_x)
    with R_w - K * z_w precomputed per output channel (``weight_rowsum``) and R_x delivered by
    the activation quantizer."""

    def __init__(self, in_features, out_features, bias=False, require_quantizer=True):
        super().__init__()
        self.in_features = in_features
        self.out_features = out_features
        self.require_quantizer = require_quantizer
        self.register_buffer("weight_scales", torch.zeros((out_features, 1), requires_grad=False, dtype=torch.float16))
        self.register_buffer("weight_zeros", torch.zeros((out_features, 1), requires_grad=False, dtype=torch.float16))
        self.register_buffer("weight_rowsum", torch.zeros((out_features,), requires_grad=False, dtype=torch.int32))
        self.register_buffer("weight", _placeholder_weight((out_features, in_features // 2), torch.uint8))
        if bias:
            self.register_buffer("bias", torch.zeros((out_features), dtype=torch.float16))
        else:
            self.bias = None
        if require_quantizer:
            self.quantizer = AsymQuantizer(shifted=True)

    _decode_spec = (_ops.EPI_ASYM_ROWSUM, (("w", "weight"), ("w_scale_1", "weight_scales"), ("w_zeros_1", "weight_zeros"),
                                           ("w_rowsum_adj", "weight_rowsum")))

    def forward(self, x):
        if self.require_quantizer:
            y = self._own_quantizer_decode(x)
            if y is not None:
                return y
            x = self._quantize(x) if self.fused else self.quantizer(x)
        assert type(x) == tensor_utils.PackedQuantizedTensor and x.rowsum_x is not None, \
            "Input should come from AsymQuantizer(shifted=True), or require_quantizer should be set"
        if self.fused and self._use_shadow(x):
            return tensor_utils.linear_forward_shadow(_ops.EPI_ASYM_ROWSUM, x.shadow_x, x.scales_x, x.zeros_x,
                                                      self.weight_shadow, self.weight_scales, self.weight_zeros,
                                                      bias=self.bias, rowsum_x=x.rowsum_x, w_rowsum_adj=self.weight_rowsum)
        if self.fused:
            return tensor_utils.linear_forward_rowsum(x.quantized_x, x.scales_x, x.zeros_x, x.rowsum_x, self.weight,
                                                      self.weight_scales, self.weight_zeros, self.weight_rowsum,
                                                      bias=self.bias,
                                                      room_bytes=self.prefill_room_bytes)
        acc = tensor_utils.matmul(x.quantized_x, self.weight)
        lead = acc.shape[:-1]
        y = _ops.asym_rowsum_dequant(acc.view(-1, acc.shape[-1]), x.scales_x, x.zeros_x, x.rowsum_x, self.weight_scales,
                                     self.weight_zeros, self.weight_rowsum, self.bias)
        return y.view(*lead, -1)

    @classmethod
    def from_linear(cls, module: torch.nn.Linear, require_quantizer: bool = True):
        """Per-output-channel min/max quantization of ``module.weight`` on the device it lives on
        (the activation quantizer kernel, applied to the weight rows)."""
        w = module.weight.data
        assert w.is_cuda, "weight preparation runs on the GPU: move the layer there first"
        new = _unfilled(cls, module.in_features, module.out_features, bias=module.bias is not None,
                        require_quantizer=require_quantizer, device=w.device)
        q, scale, zeros, rowsum = tensor_utils.quantize_asym_shifted(w.to(torch.float16).contiguous())
        new.weight.copy_(q)
        new.weight_scales.copy_(scale)
        new.weight_zeros.copy_(zeros)
        new.weight_rowsum.copy_(rowsum - module.in_features * zeros.view(-1).to(torch.int32))
        if module.bias is not None:
            new.bias.copy_(module.bias)
        return new


@native_call("own_layer")
class LinearQuant4bitDUASQRowSum(_Linear4bitBase):
    """Dual-uniform asymmetric layer with the exact zero-point correction.  Not in the reference: its
    LinearQuant4bitDUASQ (linear.py:209-297) quantizes input columns 0..9 of every weight row with one
    (scale, zero) pair and the others with a second pair, and its epilogue (src/kernels/quant2.cu:158-186) then
    applies ONE pair per output column to the whole accumulator.  Here the accumulator is split at input column 10
    and each part gets the row-sum correction with its own pair:
        y = s_x * ( s_1 * corr(k < 10) + s_2 * corr(k >= 10) ),  corr = acc - z_x * (R_w - n_k * z_w) - z_w * R_x
    Codes and zero points are stored minus 8 (the signed GEMM reads them exactly), ``weight_rowsum_1/2`` hold
    ``R_w - n_k * z_w`` of the two ranges.  The forward is one launch for up to eight rows and some hundred short ones, quantizer + GEMM with the
    epilogue inside for the shapes of the decode and prefill kernels, else quantizer, GEMM into int32, epilogue."""

    def __init__(self, in_features, out_features, bias=False, require_quantizer=True):
        super().__init__()
        self.in_features = in_features
        self.out_features = out_features
        self.require_quantizer = require_quantizer
        for k in (1, 2):
            self.register_buffer(f"weight_scales_{k}", torch.zeros((out_features, 1), requires_grad=False, dtype=torch.float16))
            self.register_buffer(f"weight_zeros_{k}", torch.zeros((out_features, 1), requires_grad=False, dtype=torch.float16))
            self.register_buffer(f"weight_rowsum_{k}", torch.zeros((out_features,), requires_grad=False, dtype=torch.int32))
        self.register_buffer("weight", _placeholder_weight((out_features, in_features // 2), torch.uint8))
        if bias:
            self.register_buffer("bias", torch.zeros((out_features), dtype=torch.float16))
        else:
            self.bias = None
        if require_quantizer:
            self.quantizer = AsymQuantizer(shifted=True)

    _decode_spec = (_ops.EPI_ASYM_DUAL_ROWSUM, (("w", "weight"), ("w_scale_1", "weight_scales_1"), ("w_zeros_1", "weight_zeros_1"),
                                                ("w_scale_2", "weight_scales_2"), ("w_zeros_2", "weight_zeros_2"),
                                                ("w_rowsum_adj", "weight_rowsum_1"), ("w_rowsum_adj_2", "weight_rowsum_2")))

    def forward(self, x):
        if self.require_quantizer:
            y = self._own_quantizer_decode(x)
            if y is not None:
                return y
            # (the 6-bit float path of this layer reads the packed codes too: shadow and codes)
            rows = x.numel() // x.shape[-1]
            x = self.quantizer(x, shadow=True if self.fused and self._fp6_pays(rows) else False)
        assert type(x) == tensor_utils.PackedQuantizedTensor and x.rowsum_x is not None, \
            "Input should come from AsymQuantizer(shifted=True), or require_quantizer should be set"
        xq = x.quantized_x
        lead = xq.shape[:-1]
        xq2 = xq.reshape(-1, xq.shape[-1])
        if self.fused and x.shadow_x is not None and self._fp6_wanted(xq2.shape[0]):
            y = _ops.linear4bit_forward_dual_rowsum_bf6(x.shadow_x.reshape(xq2.shape[0], -1), xq2, x.scales_x, x.zeros_x,
                                                        x.rowsum_x, self.weight_shadow, self.weight,
                                                        self.weight_scales_1, self.weight_zeros_1, self.weight_scales_2,
                                                        self.weight_zeros_2, self.weight_rowsum_1, self.weight_rowsum_2,
                                                        self.bias)
        elif self.fused:
            y = _ops.linear4bit_forward_dual_rowsum(xq2, x.scales_x, x.zeros_x, x.rowsum_x, self.weight,
                                                    self.weight_scales_1, self.weight_zeros_1, self.weight_scales_2,
                                                    self.weight_zeros_2, self.weight_rowsum_1, self.weight_rowsum_2,
                                                    self.bias)
        else:
            acc = _ops.matmul(xq2, self.weight)
            y = _ops.asym_dual_rowsum_dequant(acc, xq2, x.scales_x, x.zeros_x, x.rowsum_x, self.weight,
                                              self.weight_scales_1, self.weight_zeros_1, self.weight_scales_2,
                                              self.weight_zeros_2, self.weight_rowsum_1, self.weight_rowsum_2, self.bias)
        return y.view(*lead, -1)

    @classmethod
    def from_linear(cls, module: torch.nn.Linear, require_quantizer: bool = True):
        """Per-output-channel min/max quantization of input columns 0..9 and of the others, each range on its own,
        on the device the weight lives on (the activation quantizer kernel applied to the two column ranges,
        each padded with copies of its last column to a width the kernel takes: a copy changes neither the
        minimum nor the maximum)."""
        w = module.weight.data
        assert w.is_cuda, "weight preparation runs on the GPU: move the layer there first"
        K, split = module.in_features, tensor_utils.get_dual_quant_col()
        assert K > split and K % 2 == 0
        new = _unfilled(cls, K, module.out_features, bias=module.bias is not None, require_quantizer=require_quantizer,
                        device=w.device)
        w = w.to(torch.float16)
        if _ops.weight_takes_one_pass(w):
            q, ranges = _ops.weight_quant_asym(w, split, shifted=True)
            new.weight.copy_(q)
            for k, (n_k, (scale, zeros, rowsum)) in enumerate(zip((split, K - split), ranges), start=1):
                getattr(new, f"weight_scales_{k}").copy_(scale)
                getattr(new, f"weight_zeros_{k}").copy_(zeros)
                getattr(new, f"weight_rowsum_{k}").copy_(rowsum - n_k * zeros.view(-1).to(torch.int32))
            if module.bias is not None:
                new.bias.copy_(module.bias)
            return new
        codes = []
        for k, (lo, hi) in enumerate(((0, split), (split, K)), start=1):
            part = w[:, lo:hi]
            pad = (-(hi - lo)) % 32
            if pad:
                part = torch.cat([part, part[:, -1:].expand(-1, pad)], dim=1)
            q, scale, zeros, _ = tensor_utils.quantize_asym_shifted(part.contiguous())
            c = quant_utils.unpack_i4(q)[:, :hi - lo]          # signed codes
            codes.append(c)
            getattr(new, f"weight_scales_{k}").copy_(scale)
            getattr(new, f"weight_zeros_{k}").copy_(zeros)
            getattr(new, f"weight_rowsum_{k}").copy_(c.sum(dim=1, dtype=torch.int32) - (hi - lo) * zeros.view(-1).to(torch.int32))
        new.weight.copy_(quant_utils.pack_i4(torch.cat(codes, dim=1).to(torch.int8), sym=True))
        if module.bias is not None:
            new.bias.copy_(module.bias)
        return new


@native_call("sym_layer")
class Linear4bitDUSQ(_Linear4bitBase):
    """Symmetric layer with two per-row weight scales: input columns < 10 were quantized
    with scale 1, the rest with scale 2; the epilogue picks per OUTPUT column < 10
    (linear.py:147-206, quant2.cu:81)."""

    def __init__(self, in_features, out_features, bias=False, dtype=torch.float16):
        super().__init__()
        self.in_features = in_features
        self.out_features = out_features
        self.register_buffer("weight_scales_1", torch.zeros((out_features, 1), requires_grad=False))
        self.register_buffer("weight_scales_2", torch.zeros((out_features, 1), requires_grad=False))
        self.register_buffer("weight", _placeholder_weight((out_features, in_features // 2), torch.uint8))
        if bias:
            self.register_buffer("bias", torch.zeros((out_features), dtype=dtype))
        else:
            self.bias = None

    _decode_spec = (_ops.EPI_SYM_DUAL, (("w", "weight"), ("w_scale_1", "weight_scales_1"), ("w_scale_2", "weight_scales_2")))

    def forward(self, x):
        assert type(x) == tensor_utils.PackedQuantizedTensor
        if x._src is not None:  # up to 1024 rows straight from SymQuantizer: quantizer and GEMM in one library call
            y = self._take_deferred(x)
            if y is not None:
                return y
        xq, scales_x = x.quantized_x, x.scales_x
        if self.fused and self._use_shadow(x):
            return tensor_utils.linear_forward_shadow(_ops.EPI_SYM_DUAL, x.shadow_x, scales_x, None, self.weight_shadow,
                                                      self.weight_scales_1, None, self.weight_scales_2, bias=self.bias)
        if self.fused:
            return tensor_utils.linear_forward(_ops.EPI_SYM_DUAL, xq, scales_x, None, self.weight,
                                               self.weight_scales_1, None, self.weight_scales_2, bias=self.bias,
                                               room_bytes=self.prefill_room_bytes)
        acc = tensor_utils.matmul(xq, self.weight)
        return self._finish(tensor_utils.sym_dual_dequant(acc, scales_x, self.weight_scales_1, self.weight_scales_2))

    @staticmethod
    def from_float(module: torch.nn.Linear, weight_scales_1=None, weight_scales_2=None):
        w = module.weight.data
        make = Linear4bitDUSQ if weight_scales_1 is None or weight_scales_2 is None else functools.partial(_unfilled, Linear4bitDUSQ)
        new = make(module.in_features, module.out_features, bias=module.bias is not None, dtype=w.dtype).to(w.dtype)
        if weight_scales_1 is not None and weight_scales_2 is not None:
            shape = (module.out_features, 1)
            assert weight_scales_1.shape == shape, "weight_scales_1 should have shape (out_features, 1)"
            assert weight_scales_2.shape == shape, "weight_scales_2 should have shape (out_features, 1)"
            split = tensor_utils.get_dual_quant_col()
            q = _pack_given(w, lambda: torch.cat([(w[:, :split] / weight_scales_1.to(w.device)).round(),
                                                  (w[:, split:] / weight_scales_2.to(w.device)).round()], dim=-1),
                            (weight_scales_1, weight_scales_2), split)
            _store((new.weight, q), (new.weight_scales_1, weight_scales_1.to(w.dtype)),
                   (new.weight_scales_2, weight_scales_2.to(w.dtype)), *_bias_pair(new, module))
        return new


@native_call("own_layer")
class LinearQuant4bitDUASQ(_Linear4bitBase):
    """Asymmetric dual-uniform layer (linear.py:209-297)."""

    def __init__(self, in_features, out_features, bias=False, require_quantizer=True):
        super().__init__()
        self.in_features = in_features
        self.out_features = out_features
        self.require_quantizer = require_quantizer
        for name in ("weight_scales_1", "weight_zeros_1", "weight_scales_2", "weight_zeros_2"):
            self.register_buffer(name, torch.zeros((out_features, 1), requires_grad=False, dtype=torch.float16))
        self.register_buffer("weight", _placeholder_weight((out_features, in_features // 2), torch.uint8))
        if bias:
            self.register_buffer("bias", torch.zeros((out_features), dtype=torch.float16))
        else:
            self.bias = None
        if self.require_quantizer:
            self.quantizer = AsymQuantizer()

    _decode_spec = (_ops.EPI_ASYM_DUAL, (("w", "weight"), ("w_scale_1", "weight_scales_1"), ("w_zeros_1", "weight_zeros_1"),
                                         ("w_scale_2", "weight_scales_2"), ("w_zeros_2", "weight_zeros_2")))

    def forward(self, x):
        if self.require_quantizer:
            y = self._own_quantizer_decode(x)
            if y is not None:
                return y
            x = self._quantize(x) if self.fused else self.quantizer(x)
        assert type(x) == tensor_utils.PackedQuantizedTensor, \
            "Input should be quantized tensor, or require_quantizer should be passed as initial argument"
        xq, scales_x, zeros_x = x.quantized_x, x.scales_x, x.zeros_x
        if self.fused and self._use_shadow(x):
            return tensor_utils.linear_forward_shadow(_ops.EPI_ASYM_DUAL, x.shadow_x, scales_x, zeros_x,
                                                      self.weight_shadow, self.weight_scales_1, self.weight_zeros_1,
                                                      self.weight_scales_2, self.weight_zeros_2, bias=self.bias)
        if self.fused:
            return tensor_utils.linear_forward(_ops.EPI_ASYM_DUAL, xq, scales_x, zeros_x, self.weight,
                                               self.weight_scales_1, self.weight_zeros_1, self.weight_scales_2,
                                               self.weight_zeros_2, bias=self.bias,
                                               room_bytes=self.prefill_room_bytes)
        acc = tensor_utils.matmul(xq, self.weight)
        return self._finish(tensor_utils.asym_dual_dequant(acc, scales_x, zeros_x, self.weight_scales_1,
                                                           self.weight_zeros_1, self.weight_scales_2,
                                                           self.weight_zeros_2))

    @classmethod
    def from_linear(cls, module: torch.nn.Linear, require_quantizer=True):
        new = _unfilled(cls, module.in_features, module.out_features, bias=module.bias is not None,
                        require_quantizer=require_quantizer)
        w = module.weight.data
        split = tensor_utils.get_dual_quant_col()
        if _ops.weight_takes_one_pass(w):
            q, ((s1, z1), (s2, z2)) = _ops.weight_quant_asym(w, split)
        else:
            s1, z1, c1 = _asym_params(w[:, :split])
            s2, z2, c2 = _asym_params(w[:, split:])
            q = quant_utils.pack_i4(torch.cat([c1, c2], dim=-1).to(torch.int8), sym=False)
        _store((new.weight, q), (new.weight_scales_1, s1.to(torch.float16)), (new.weight_zeros_1, z1.to(torch.float16)),
               (new.weight_scales_2, s2.to(torch.float16)), (new.weight_zeros_2, z2.to(torch.float16)), *_bias_pair(new, module))
        return new


@native_call("eight_bit")
class LinearQuant8bitASQ(_MovesTogether):
    """Asymmetric 8-bit linear layer on float32 activations (linear.py:300-368): buffers ``weight`` int8
    [N, K] (codes 0..127), ``weight_scales`` / ``weight_zeros`` float32 [N, 1], optional ``bias``
    float32 [N]; float32 result.  ``fused = False`` runs the reference's three steps (same bits)."""

    fused = True
    # the fused forward reads a copy of ``weight`` arranged for the MFMA operand layout (as many bytes again; not
    # part of the state_dict; rebuilt when ``weight`` changes).  tiled = False reads ``weight`` itself: same bits,
    # about half the speed on large inputs; so does a layer whose weight was made in torch.inference_mode(): such a
    # tensor counts no versions, and a copy could not follow its changes
    tiled = True
    _tiled_key = None

    def _tiled_weight(self):
        """The copy of ``weight`` for the fused forward, None for a layer that reads ``weight`` itself."""
        if not self.tiled or self.weight.is_inference():
            return None
        if self._tiled_stale():
            with _copying:
                if self._tiled_stale():
                    _put_copy(self, "weight_tiled", "_tiled_key", tensor_utils.weight_tile_8bit, True)
        return self.weight_tiled

    def _tiled_stale(self):
        return self._tiled_key != _weight_key(self) or self._buffers.get("weight_tiled") is None

    def __init__(self, in_features, out_features, bias=False, require_quantizer=True):
        super().__init__()
        self.in_features = in_features
        self.out_features = out_features
        self.require_quantizer = require_quantizer
        self.register_buffer("weight_scales", torch.zeros((out_features, 1), requires_grad=False, dtype=torch.float32))
        self.register_buffer("weight_zeros", torch.zeros((out_features, 1), requires_grad=False, dtype=torch.float32))
        self.register_buffer("weight", _placeholder_weight((out_features, in_features), torch.int8))
        if bias:
            self.register_buffer("bias", torch.zeros((out_features), dtype=torch.float32))
        else:
            self.bias = None
        if require_quantizer:
            self.quantizer = AsymQuantizer8bit()

    # rows up to which the layer's own quantizer and the GEMM go through one library call (a step of a few rows
    # costs more on the host than on the GPU; larger inputs hide the second call behind the first launch)
    one_call_rows = 1024

    def forward(self, x):
        if self.require_quantizer:
            if self.fused and type(x) is torch.Tensor and x.dtype is torch.float32 and x.is_cuda and x.is_contiguous() \
                    and x.shape[-1] == self.in_features and self.in_features % 32 == 0 and x.data_ptr() % 16 == 0 \
                    and 0 < x.numel() <= self.one_call_rows * self.in_features and type(self.quantizer) is AsymQuantizer8bit \
                    and self.quantizer.fused:
                return _ops.quantize_linear8bit_forward(x, self.weight, self._tiled_weight(), self.weight_scales,
                                                        self.weight_zeros, self.bias)
            x = self.quantizer(x)
        assert type(x) == tensor_utils.PackedQuantizedTensor, \
            "Input should be quantized tensor, or require_quantizer should be passed as initial argument"
        xq, scales_x, zeros_x = x.quantized_x, x.scales_x, x.zeros_x
        rows = xq.numel() // xq.shape[-1] if xq.shape[-1] else 0
        # up to four rows (two for rows longer than 4096 elements) run a kernel that reads `weight` itself
        few_rows = rows <= 4 and self.in_features <= (8192 if rows <= 2 else 4096)
        copy = self._tiled_weight() if self.fused and not few_rows else None
        if copy is not None:
            return tensor_utils.linear8bit_forward(xq, scales_x, zeros_x, copy, self.weight_scales,
                                                   self.weight_zeros, self.bias, tiled_rows=self.out_features)
        if self.fused:
            return tensor_utils.linear8bit_forward(xq, scales_x, zeros_x, self.weight, self.weight_scales,
                                                   self.weight_zeros, self.bias)
        acc = tensor_utils.matmul_8bit(xq, self.weight)
        y = tensor_utils.asym_dequant_hprec(acc, scales_x, zeros_x, self.weight_scales, self.weight_zeros)
        return y if self.bias is None else y + self.bias

    @classmethod
    def from_linear(cls, module: torch.nn.Linear, require_quantizer: bool = True):
        """Per-row scale / zero over |W| with 127 steps, codes clamp(round(W / s) + z, 0, 127)
        (linear.py:338-368)."""
        new = _unfilled(cls, module.in_features, module.out_features, bias=module.bias is not None,
                        require_quantizer=require_quantizer)
        w = module.weight.data
        if _ops.weight_takes_one_pass(w, torch.float32):
            q, scale, zeros = _ops.weight_quant_asym_8bit(w)
        else:
            levels = 2 ** 7
            aw = w.abs()
            w_max = aw.amax(dim=-1, keepdim=True)
            w_min = aw.amin(dim=-1, keepdim=True)
            scale = (w_max - w_min) / (levels - 1)
            zeros = (-w_min / scale).round().to(torch.float32)
            q = torch.clamp(torch.round(w / scale) + zeros, 0, levels - 1).to(torch.int8)
        _store((new.weight, q), (new.weight_scales, scale.to(torch.float32)), (new.weight_zeros, zeros.to(torch.float32)),
               *_bias_pair(new, module))
        return new
