"""PyTorch-ROCm front end of the C ABI: a registered operator and a drop-in linear layer.

  torch.ops.lutgemm.matvec(x, handle)   y[..., n] = x[..., k] @ W  for a packed BCQ weight
  LutLinear                             nn.Module around one packed weight (+ optional bias)

The operator launches on torch's current stream and allocates nothing but its output (and, when more than 16
rows first need it, the handle's room for partial sums, which capture allows), so it can
be captured into a HIP graph like any other torch op once it has run on the capturing stream.  Batches larger than `dense_threshold`
rows go through the dequantised fp16 weight and the library GEMM, the route the reference takes
for every m > 1 (lutGEMM/src/kernels.cu:73-79).  Like the reference, which dequantises into one
grow-only scratch buffer of the process on every such call (lutGEMM/src/cuda/tmpWeight.hpp:28-35,
lutGEMM/src/nQWeight_fp16.cu:93-99), the dense weight is rebuilt per call in a scratch buffer shared
by all layers (one per device and stream), so a layer never holds more than its packed weight;
`keep_dense=True` keeps a private dense copy instead (2 k n bytes) and skips the rebuild.  Up to
the threshold the library streams the packed weight
(one or two rows through the table-lookup kernels, 3 to 16 through the kernel for few rows, more through the kernel
for many rows).  The default threshold depends on the weight and on keep_dense (default_dense_threshold):
it is where the two routes met when measured on MI355X.
"""


def default_dense_threshold(weight, keep_dense=False):
    """Rows up to which the packed route beats dequantised weight + library GEMM (measured on MI355X
    at k = n = 12288 and at k = 7168, n = 28672; LutLinear(dense_threshold=...) overrides).

    The lines come from passes of the batch kernel, which layers took when they were drawn: up to 16 rows at
    22 / 24 / 30 / 36 us for one to four planes and 41 / 43 / 50 / 57 us for five to eight (k = n = 12288).  The dense route costs the
    dequantisation (75 us up to four planes, 97-130 us for five to eight) plus the GEMM (50-56 us up
    to 32 rows), so by default it only pays from the number of passes on that costs as much:
    80 rows for one or two planes, 64 for three, 48 beyond.  A layer that keeps its dense copy
    (keep_dense) pays the GEMM alone: 32 rows for one or two planes, 16 for three to seven, and
    eight planes leave the packed route from three rows on (57 against 50 us).

    3 to 16 rows take the kernel for few rows by now (12288 x 12288, two planes, 8 rows 18 us; four planes, 16 rows 32) and more
    no longer take passes of 16, so the packed route would stay ahead for longer (12288 x 12288, three planes, 160 rows: 130
    against 192 us).  The lines are kept all the same, because the routes are not interchangeable: the dense one passes gradients to x, follows autocast, can be captured on a stream that has not
    launched on the handle, and rounds the weight to fp16, so its results differ by some 4e-4 of their norm."""
    q = weight.nb
    if keep_dense:
        return 32 if q <= 2 else 16 if q <= 7 else 2
    return 80 if q <= 2 else 64 if q == 3 else 48


import weakref

import numpy as np
import torch
from torch.autograd import forward_ad

from . import BCQWeight, LutGemmError, ERR_BAD_SHAPE, MAX_BATCH

_weights = weakref.WeakValueDictionary()  # operator argument (an int) -> BCQWeight
_next_id = [1]
_dense_scratch = {}   # (device index, stream handle) -> grow-only fp16 buffer for dequantised weights


def dense_scratch(halves, device, stream_handle):
    """View of `halves` fp16 elements of the process-wide scratch buffer of (device, stream); the
    buffer only ever grows (the counterpart of the reference's tmpWeight singleton)."""
    key = (device.index, stream_handle)
    buf = _dense_scratch.get(key)
    if buf is None or buf.numel() < halves:
        buf = torch.empty(halves, dtype=torch.float16, device=device)
        _dense_scratch[key] = buf
    return buf[:halves]


def register(weight):
    """Make a BCQWeight addressable by the operator; returns its integer handle."""
    hid = _next_id[0]
    _next_id[0] += 1
    _weights[hid] = weight
    return hid


def _lookup(handle):
    w = _weights.get(int(handle))
    if w is None:
        raise LutGemmError(ERR_BAD_SHAPE, "operator handle %d is not registered (or its weight was freed)" % handle)
    return w


def _launch(x, handle, bias):
    w = _lookup(handle)
    if not x.is_cuda or x.dtype != torch.float16:
        raise TypeError("lutgemm::matvec needs a float16 tensor on the GPU, got %s on %s" % (x.dtype, x.device))
    k, n = w.kSize, w.mSize
    if x.shape[-1] != k:
        raise LutGemmError(ERR_BAD_SHAPE, "last dimension %d != k %d" % (x.shape[-1], k))
    if bias is not None and (bias.dtype != torch.float16 or bias.device != x.device or bias.shape != (n,) or not bias.is_contiguous()):
        raise LutGemmError(ERR_BAD_SHAPE, "the bias has to be a contiguous float16 [%d] on %s" % (n, x.device))
    device = x.device
    if torch.cuda.current_device() != device.index:
        with torch.cuda.device(device):
            return _launch(x, handle, bias)
    flat = x.dim() == 2
    x2 = x if flat and x.is_contiguous() else x.reshape(-1, k).contiguous()
    m = x2.shape[0]
    y = torch.empty((m, n), dtype=torch.float16, device=device)
    stream = _raw_stream(device.index)
    xp, yp, bp = x2.data_ptr(), y.data_ptr(), 0 if bias is None else bias.data_ptr()
    for r0 in range(0, m, MAX_BATCH):
        w.matvec_bias(xp + 2 * k * r0, yp + 2 * n * r0, bp, min(MAX_BATCH, m - r0), stream)
    return y if flat else y.reshape(x.shape[:-1] + (n,))


def _raw_stream(index):
    return torch.cuda.current_stream(index).cuda_stream


# the stream's handle without a Stream object around it, where torch has that (1.5 us less per call)
_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", _raw_stream)


@torch.library.custom_op("lutgemm::matvec", mutates_args=())
def matvec(x: torch.Tensor, handle: int) -> torch.Tensor:
    return _launch(x, handle, None)


@matvec.register_fake
def _(x, handle):
    w = _lookup(handle)
    return x.new_empty(x.shape[:-1] + (w.mSize,))


@torch.library.custom_op("lutgemm::matvec_bias", mutates_args=())
def matvec_bias(x: torch.Tensor, handle: int, bias: torch.Tensor) -> torch.Tensor:
    return _launch(x, handle, bias)


@matvec_bias.register_fake
def _(x, handle, bias):
    w = _lookup(handle)
    return x.new_empty(x.shape[:-1] + (w.mSize,))


_transformed = getattr(torch._C._functorch, "is_functorch_wrapped_tensor", lambda bias: True)


def _joins_call(bias, x, n):
    """Whether the bias may go with the call, which treats it as a constant: float16 [n] on x's device, and neither
    differentiated (in reverse or forward mode), mapped over nor traced (a compiler fuses an addition by itself)."""
    return (bias.dtype == torch.float16 and bias.shape == (n,) and bias.device == x.device and not bias.requires_grad
            and not torch.compiler.is_compiling() and type(bias) in (torch.Tensor, torch.nn.Parameter) and not _transformed(bias)
            and forward_ad.unpack_dual(bias).tangent is None and bias.is_contiguous())


class LutLinear(torch.nn.Module):
    """y = x @ W (+ bias) with W held as a packed BCQ weight on the current device.

    container: dict(bW, alpha, q_bias, k, n, q, num_groups) as quantize.to_container returns.
    """

    def __init__(self, container, bias=None, dense_threshold=None, autotune=False, keep_dense=False):
        super().__init__()
        c = container
        self.device = torch.device("cuda", torch.cuda.current_device())   # the packed weight lives here
        self.keep_dense = keep_dense
        self.weight = BCQWeight(c["bW"], c["alpha"], c["k"], c["n"], c["q"], c["num_groups"], c.get("q_bias"))
        if autotune:
            self.weight.autotune(torch.cuda.current_stream().cuda_stream)
        self.handle = register(self.weight)
        self.in_features, self.out_features = c["k"], c["n"]
        self.dense_threshold = default_dense_threshold(self.weight, keep_dense) if dense_threshold is None else dense_threshold
        self._dense = None
        if bias is not None:
            self.register_buffer("bias", torch.as_tensor(bias).to(torch.float16).to(self.device))
        else:
            self.bias = None

    @classmethod
    def from_file(cls, path, bias=None, **kw):
        self = cls.__new__(cls)
        torch.nn.Module.__init__(self)
        self.device = torch.device("cuda", torch.cuda.current_device())
        self.keep_dense = kw.get("keep_dense", False)
        self.weight = BCQWeight.load(path)
        if kw.get("autotune", False):
            self.weight.autotune(torch.cuda.current_stream().cuda_stream)
        self.handle = register(self.weight)
        self.in_features, self.out_features = self.weight.kSize, self.weight.mSize
        dt = kw.get("dense_threshold")
        self.dense_threshold = default_dense_threshold(self.weight, self.keep_dense) if dt is None else dt
        self._dense = None
        if bias is not None:
            self.register_buffer("bias", torch.as_tensor(bias).to(torch.float16).to(self.device))
        else:
            self.bias = None
        return self

    @classmethod
    def from_linear(cls, linear, qbits, group_size=128, method="rtn", rounds=15, **kw):
        """Quantise a torch.nn.Linear (weight [out, in]) and pack it."""
        from . import quantize
        c, _ = quantize.quantize_linear(linear.weight.detach().float(), qbits, group_size, method, rounds)
        b = None if linear.bias is None else linear.bias.detach()
        return cls(c, bias=b, **kw)

    def dense_weight(self):
        """Dequantised fp16 weight on the layer's device as W^T [n][k], the orientation the
        dequantise kernel writes in 1 KiB runs.  Rebuilt on torch's current stream into the shared
        scratch buffer of that stream on every call (valid until the next layer's call on the
        stream); with keep_dense it is built once and kept by the layer."""
        if self._dense is not None:
            return self._dense
        stream = torch.cuda.current_stream(self.device).cuda_stream
        if self.keep_dense:
            Wt = torch.empty((self.out_features, self.in_features), dtype=torch.float16, device=self.device)
        else:
            Wt = dense_scratch(self.out_features * self.in_features, self.device, stream).view(self.out_features, self.in_features)
        with torch.cuda.device(self.device):
            self.weight.dequantize(Wt.data_ptr(), True, stream)
        if self.keep_dense:
            self._dense = Wt
        return Wt

    def forward(self, x):
        """The bias is added to the float16 result.  On the packed route it goes with the call, which gives the same bits,
        where it is what the constructor made of it (_joins_call)."""
        rows = x.numel() // x.shape[-1]
        if x.dtype != torch.float16:
            x = x.to(torch.float16)
        bias = self.bias
        if rows > self.dense_threshold:
            y = torch.nn.functional.linear(x, self.dense_weight())
        elif bias is not None and _joins_call(bias, x, self.out_features):
            return torch.ops.lutgemm.matvec_bias(x, self.handle, bias)
        else:
            y = torch.ops.lutgemm.matvec(x, self.handle)
        return y if bias is None else y + bias


def container_from_numpy(bW, alpha, k, n, q, num_groups, q_bias=None):
    return dict(bW=np.asarray(bW), alpha=np.asarray(alpha), q_bias=q_bias, k=k, n=n, q=q, num_groups=num_groups)
