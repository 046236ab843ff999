"""Caller-side conveniences around the linear-layer path: a torch module that owns native-layout weights, and a small
on-disk container for them.  (The reference leaves both to the framework that embeds it -- DeepSpeed, README.md:19.)"""
import json
import struct

import numpy as np
import torch

from . import quant
from . import (MI355X_CUS, group_exps_bytes, heuristic_splitk_mi355x, linear_forward_native, native_bytes, pack_group_exps, to_native,
               weight_dequant_native_cuda, weight_prepacking_native_cpu, weight_quantize_native_cuda)

_MAGIC = b"FP6MI\x00\x01\x00"   # name, NUL, layout version 1, reserved


_peek_transform = getattr(getattr(torch._C, "_functorch", None), "peek_interpreter_stack", None)
_dispatch_modes = getattr(torch._C, "_len_torch_dispatch_stack", None)


def _values_only(t):
    """Whether nothing but t's values counts in what is done with it: no derivative, transform, trace, subclass or dispatch mode has a part in it, which a kernel
    that is handed t's address would pass by.  (A torch that lacks one of the names asked here is taken to have one of these active.)"""
    return (type(t) in (torch.Tensor, torch.nn.Parameter) and not (t.requires_grad and torch.is_grad_enabled())
            and _peek_transform is not None and _peek_transform() is None and getattr(torch.autograd.forward_ad, "_current_level", 0) < 0
            and _dispatch_modes is not None and _dispatch_modes() == 0 and not torch.jit.is_tracing() and not t.is_neg())


class _AutoRows(int):
    """What dequant_above reads under "auto": the number of rows, and "auto" again for a module that it is assigned to.  (Modules that library version 139
    pickled whole hold one.)"""


_CROSSOVER, _CROSSOVER_LIBRARY = 32768, 3072   # FPxLinear.PREFILL_CROSSOVER as it is shipped, and the one without the wide tiles


class FPxLinear(torch.nn.Module):
    """y = x @ dequant(W)^T (+ bias) with W held in the native gfx950 layout.  Weights are buffers, not parameters:
    the layer is inference-only, like the kernels."""

    # Batch size from which dequantize + FP16 library GEMM is no slower than the mixed-input kernels, measured through this module at 4096^2, 8192^2, 28672x8192,
    # 8192x28672, 11008x4096, 1024x8192, 1024^2, 4608x4544 and 2560x18944, FP6 with row scales and FP5 with group exponents.  Kernel time / time of dequantization +
    # library GEMM: 0.33-0.99 at 3072 rows, 0.35-1.06 at 4096, 0.40-0.99 at 4100, 0.44-1.07 at 6144, 0.51-1.06 at 8192, 0.73-1.03 at 16384, 0.85-1.10 at 32768
    # (8192^2 at 4096 rows 369 us against 394, at 16384 1465 against 1464); with a bias, which the kernels add by themselves, 0.29-1.03 at 4096 and 0.58-0.96 at
    # 16384.  That is with the wide tiles, so on 256 CUs and with K up to 2^20; without them the two cross at 3072 rows.
    PREFILL_CROSSOVER = _CROSSOVER

    def __init__(self, in_features, out_features, exponent=3, mantissa=2, bias=None, split_k=None, dequant_above="auto", group_scales=False):
        """split_k: number of pieces of K, None for the heuristic's choice; under dequant_above="auto" it holds for less than 3072 rows.
        group_scales: the layer also holds one exponent byte per row and 128 columns (factor 1 until weights are loaded).
        dequant_above: batch size from which forward() dequantizes the weights to a temporary fp16 matrix on the GPU and calls
        the FP16 library GEMM instead (the temporary costs 2 bytes per weight for the duration of the call).  None never does; an
        integer sets the threshold; "auto" (default) is PREFILL_CROSSOVER rows, or 3072 where the wide tiles do not run.  Under "auto" an
        input of 3072 rows or more that the kernels cannot take as it is (_kernels_take: one that requires a gradient, say) also goes through
        the library.  A module that a version up to 138 pickled whole holds the number that "auto" was then, 3072."""
        super().__init__()
        self.dequant_above = dequant_above
        if out_features % 256 or in_features % 64:
            raise ValueError("FPxLinear needs out_features %% 256 == 0 and in_features %% 64 == 0")
        self.in_features, self.out_features = in_features, out_features
        self.exponent, self.mantissa = exponent, mantissa
        self.split_k = split_k
        self._split_cache = {}
        self.register_buffer("weight_native", torch.zeros(native_bytes(exponent, mantissa, out_features, in_features) // 4, dtype=torch.int32))
        self.register_buffer("scales", torch.ones(out_features, dtype=torch.float16))
        self.register_buffer("bias", bias)
        # per-group exponents (one byte per row and 128 columns, in the kernels' order), or None for row scales only
        self.register_buffer("group_exps", torch.full((group_exps_bytes(out_features, in_features),), 127, dtype=torch.uint8) if group_scales else None)

    @classmethod
    def from_raw(cls, raw_int32, scales, exponent=3, mantissa=2, bias=None, split_k=None):
        """raw_int32: the reference's raw weight tensor [OC, IC/32*x] (CPU); scales: float16 [OC]."""
        x = 1 + exponent + mantissa
        OC, IC = raw_int32.shape[0], raw_int32.shape[1] * 32 // x
        m = cls(IC, OC, exponent, mantissa, bias, split_k)
        m.weight_native.copy_(weight_prepacking_native_cpu(exponent, mantissa, raw_int32))
        m.scales.copy_(scales)
        return m

    @classmethod
    def from_prepacked(cls, packed_int32, scales, exponent=3, mantissa=2, bias=None, split_k=None):
        """packed_int32: output of weight_prepacking*_cpu (the reference layout), on CPU or GPU."""
        x = 1 + exponent + mantissa
        OC, IC = packed_int32.shape[0], packed_int32.shape[1] * 32 // x
        m = cls(IC, OC, exponent, mantissa, bias, split_k).to(packed_int32.device)
        m.weight_native.copy_(to_native(packed_int32, exponent, mantissa))
        m.scales.copy_(scales.to(packed_int32.device))
        return m

    @classmethod
    def from_float(cls, weight, exponent=3, mantissa=2, bias=None, split_k=None, group_scales=False):
        """Quantizes a float [OC, IC] weight row-wise (round to nearest even, absmax scales) and packs it; a weight that
        already lives on the GPU is quantized there (same bits as the host path).  group_scales=True adds a power-of-two
        factor per row and 128 columns (quant.quantize_groupwise), which the conversion instruction applies."""
        on_gpu = weight.device.type == "cuda" and weight.dtype in (torch.float16, torch.bfloat16, torch.float32)
        if group_scales and on_gpu:
            native, scales, gexp = weight_quantize_native_cuda(exponent, mantissa, weight.detach(), True)
            m = cls(weight.shape[1], weight.shape[0], exponent, mantissa, bias, split_k).to(weight.device)
            m.weight_native.copy_(native)
            m.scales.copy_(scales)
            m.group_exps = gexp
            return m
        if group_scales:
            codes, scales, exps = quant.quantize_groupwise(weight.detach().float().cpu().numpy(), exponent, mantissa)
            raw = torch.from_numpy(quant.pack_raw(codes, exponent, mantissa))
            m = cls.from_raw(raw, torch.from_numpy(scales), exponent, mantissa, bias, split_k)
            m.group_exps = pack_group_exps(torch.from_numpy(exps), weight.shape[0], weight.shape[1])
            return m.to(weight.device)
        if weight.device.type == "cuda" and weight.dtype in (torch.float16, torch.bfloat16, torch.float32):
            native, scales = weight_quantize_native_cuda(exponent, mantissa, weight.detach())
            m = cls(weight.shape[1], weight.shape[0], exponent, mantissa, bias, split_k).to(weight.device)
            m.weight_native.copy_(native)
            m.scales.copy_(scales)
            return m
        codes, scales = quant.quantize_rowwise(weight.detach().float().cpu().numpy(), exponent, mantissa)
        raw = torch.from_numpy(quant.pack_raw(codes, exponent, mantissa))
        return cls.from_raw(raw, torch.from_numpy(scales), exponent, mantissa, bias, split_k)

    @classmethod
    def fused(cls, layers, split_k=None):
        """One layer that computes several layers over the same input in a single launch (fused QKV, gate + up): its output
        is the concatenation of theirs along the feature axis.  Rows are independent in the native layout (16-row tiles
        are stored one after another), so fusing is a concatenation of the weight buffers, scales and biases."""
        layers = list(layers)
        first = layers[0]
        for l in layers:
            if (l.in_features, l.exponent, l.mantissa) != (first.in_features, first.exponent, first.mantissa):
                raise ValueError("fused layers must share in_features and the weight format")
            if (l.bias is None) != (first.bias is None):
                raise ValueError("fused layers must all have a bias or all have none")
            if l.weight_native.device != first.weight_native.device:
                raise ValueError("fused layers must live on one device")
            if (l.group_exps is None) != (first.group_exps is None):
                raise ValueError("fused layers must all have group exponents or all have none")
        bias = None if first.bias is None else torch.cat([l.bias for l in layers])
        m = cls(first.in_features, sum(l.out_features for l in layers), first.exponent, first.mantissa, bias, split_k)
        m = m.to(first.weight_native.device)
        m.weight_native.copy_(torch.cat([l.weight_native for l in layers]))
        m.scales.copy_(torch.cat([l.scales for l in layers]))
        if first.group_exps is not None:   # [row tile][K block][16][2] bytes: row tiles follow each other like the weights
            m.group_exps = torch.cat([l.group_exps for l in layers])
        return m

    def __getattr__(self, name):
        """nn.Module's, but that a buffer, of which a forward pass reads four, is looked for first (a call of a module with small kernels 7.9 -> 6.7 us)."""
        if name != "_buffers":   # (asked before nn.Module has made it, while a module is copied or unpickled)
            try:
                return self._buffers[name]
            except (KeyError, AttributeError):
                pass
        return super().__getattr__(name)

    def _wide_tiles(self, device):
        return self.in_features <= 1 << 20 and (device.type != "cuda" or torch.cuda.get_device_properties(device).multi_processor_count == MI355X_CUS)

    @property
    def dequant_above(self):
        """Rows from which forward() dequantizes an input that the kernels could take, on the weights' device; None: never."""
        if not self._auto:
            return self._rows
        return _AutoRows(self._rows if self._wide_tiles(self.weight_native.device) else _CROSSOVER_LIBRARY)

    @dequant_above.setter
    def dequant_above(self, rows):
        if isinstance(rows, str) and rows == "auto":   # (a subclass or a program with a PREFILL_CROSSOVER of its own means that number, whatever the device)
            rows = _AutoRows(_CROSSOVER) if self.PREFILL_CROSSOVER == _CROSSOVER else self.PREFILL_CROSSOVER
        self._auto = type(rows) is _AutoRows
        self._rows = _CROSSOVER if self._auto else rows

    def __setstate__(self, state):
        super().__setstate__(state)
        if "dequant_above" in self.__dict__:   # pickled whole when it was a plain attribute
            self.dequant_above = self.__dict__.pop("dequant_above")

    def _bias_in_kernel(self, x2):
        """Whether the kernels add the bias (to their float32 sums; otherwise a torch addition follows): a plain fp16 vector on the GPU that nothing
        differentiates or maps over."""
        b = self.bias
        return (b is not None and _values_only(b) and b.dtype == torch.float16 and b.shape == (self.out_features,) and b.is_contiguous() and b.device == x2.device)

    def _kernels_take(self, x2):
        """Whether a long prompt can leave torch.nn.functional.linear for the mixed-input kernels and nothing is lost: they are no part of an autograd graph, a
        trace or a transform, give fp16 whatever autocast would, and read contiguous rows at a 16-byte boundary; and only the wide tiles are faster."""
        kind = x2.device.type
        return (self._wide_tiles(x2.device) and _values_only(x2) and (not torch.is_autocast_enabled(kind) or torch.get_autocast_dtype(kind) == torch.float16)
                and (not x2.is_contiguous() or x2.data_ptr() % 16 == 0))

    def forward(self, x):
        # (two reshapes to the shapes at hand take 0.7 us each; a trace, whose sizes are no plain numbers, keeps them)
        shape = x.shape
        plain = type(x) is torch.Tensor and len(shape) == 2 and type(shape[1]) is int and shape[1] == self.in_features
        x2 = x if plain else x.reshape(-1, self.in_features)
        if x2.dtype != torch.float16:
            x2 = x2.half()
        rows, n = self._rows, x2.shape[0]
        if rows is not None and (n >= rows or (self._auto and n >= _CROSSOVER_LIBRARY and not self._kernels_take(x2))):
            w16 = weight_dequant_native_cuda(self.exponent, self.mantissa, self.weight_native, self.scales, self.out_features, self.in_features,
                                             self.group_exps)
            y = torch.nn.functional.linear(x2, w16)
            del w16
            if self.bias is not None:
                y = y + self.bias
            return y if plain else y.reshape(*shape[:-1], self.out_features)
        sk = self.split_k
        if not sk or (self._auto and n >= _CROSSOVER_LIBRARY):   # the heuristic's answer per batch size is remembered: the layer is called once per token
            # (split_k is for the batches up to 3071 rows; the partial sums of a long prompt would take gigabytes)
            sk = self._split_cache.get(n)
            if sk is None:
                sk = self._split_cache[n] = heuristic_splitk_mi355x(self.out_features, n, self.in_features, MI355X_CUS, self.exponent, self.mantissa)
        bias = self.bias   # (a buffer, found by nn.Module.__getattr__ in half a microsecond: read once)
        OC, fused = self.out_features, bias if bias is not None and self._bias_in_kernel(x2) else None
        y = linear_forward_native(self.exponent, self.mantissa, x2, self.weight_native, self.scales, OC, sk, None, None, self.group_exps, fused)
        if bias is not fused:
            y = y + bias
        return y if plain else y.reshape(*shape[:-1], OC)

    def extra_repr(self):
        return "in_features=%d, out_features=%d, format=e%dm%d" % (self.in_features, self.out_features, self.exponent, self.mantissa)


def save_native(path, native_int32, scales, exponent, mantissa, out_features, in_features, group_exps=None):
    """One weight matrix in the native layout: magic, little-endian uint32 header length, JSON header, native bytes, fp16 scales,
    then the packed group exponents if the weight has them."""
    nat = native_int32.detach().cpu().contiguous().numpy()
    sc = scales.detach().cpu().contiguous().numpy().astype(np.float16)
    if nat.nbytes != native_bytes(exponent, mantissa, out_features, in_features) or sc.shape != (out_features,):
        raise ValueError("buffers do not match the stated shape")
    ge = None
    if group_exps is not None:
        ge = group_exps.detach().cpu().contiguous().numpy()
        if ge.dtype != np.uint8 or ge.size != group_exps_bytes(out_features, in_features):
            raise ValueError("group_exps does not match the stated shape")
    header = json.dumps({"exponent": exponent, "mantissa": mantissa, "out_features": out_features, "in_features": in_features,
                         "layout": "native-v1", "native_bytes": int(nat.nbytes), "group_exps_bytes": 0 if ge is None else int(ge.size)}).encode()
    with open(path, "wb") as f:
        f.write(_MAGIC)
        f.write(struct.pack("<I", len(header)))
        f.write(header)
        f.write(nat.tobytes())
        f.write(sc.tobytes())
        if ge is not None:
            f.write(ge.tobytes())


def load_native(path):
    """Returns (native int32 tensor, float16 scales, header dict); the packed group exponents, if the file has them, are
    hdr["group_exps"] (uint8 tensor).  Plain binary parsing; nothing in the file is executed."""
    with open(path, "rb") as f:
        if f.read(len(_MAGIC)) != _MAGIC:
            raise ValueError("%s is not a native FPx weight file (or has another layout version)" % path)
        (hlen,) = struct.unpack("<I", f.read(4))
        if hlen > 1 << 16:
            raise ValueError("implausible header length")
        hdr = json.loads(f.read(hlen).decode())
        want = native_bytes(hdr["exponent"], hdr["mantissa"], hdr["out_features"], hdr["in_features"])
        if hdr.get("layout") != "native-v1" or hdr.get("native_bytes") != want:
            raise ValueError("header does not describe a native-v1 weight of that shape")
        nat = np.frombuffer(f.read(want), dtype=np.int32)
        sc = np.frombuffer(f.read(2 * hdr["out_features"]), dtype=np.float16)
        if nat.nbytes != want or sc.size != hdr["out_features"]:
            raise ValueError("file is truncated")
        gbytes = int(hdr.get("group_exps_bytes", 0))
        if gbytes:
            if gbytes != group_exps_bytes(hdr["out_features"], hdr["in_features"]):
                raise ValueError("header does not describe the group exponents of that shape")
            ge = np.frombuffer(f.read(gbytes), dtype=np.uint8)
            if ge.size != gbytes:
                raise ValueError("file is truncated")
            hdr["group_exps"] = torch.from_numpy(ge.copy())
    return torch.from_numpy(nat.copy()), torch.from_numpy(sc.copy()), hdr
