"""Per-timestep synapses on (N, C, H, W, T) tensors over the C ABI of ``libslayer_hip.so``.

The reference's ``_convLayer`` / ``_poolLayer`` / ``_convTransposeLayer`` / ``_unpoolLayer`` call
``F.conv3d`` / ``F.conv_transpose3d`` with a kernel of time extent 1 (src/slayer.py:499-507,
:565-575, :631-643, :732-748) and leave the gradients to autograd.  Here the operation and its
two gradients are three extension-level functions on T-innermost tensors, tied together by
``synapseConv`` / ``synapseConvTranspose`` (autograd Functions with the argument meaning of the
torch calls they replace).  There is no CPU path: tensors must live on the GPU.
"""
import ctypes
import functools

import torch

from . import _lib
from ._function import Function
from ._lib import host
from .slayerCuda import _check_device, _check_input, _on_device_of, _ptr

__all__ = ["conv", "convGradInput", "convGradWeight", "outShape", "supported", "synapseConv", "synapseConvTranspose",
           "denseEvents", "denseEventsGradWeight", "denseEventsSupported", "synapseDenseEvents", "denseRows",
           "denseRowsSupported", "denseRowsPays", "synapseDenseRows", "denseRowsGradWeight",
           "denseRowsGradWeightSupported", "pool", "poolGradInput", "synapsePool",
           "denseThin", "denseThinGradInput", "denseThinGradWeight", "synapseDenseThin"]


def _pair(v, name):
    if isinstance(v, int):
        return v, v
    v = tuple(int(x) for x in v)
    if len(v) == 3 and name != "kernel":          # torch-style triple with the time entry last
        v = v[:2]
    if len(v) != 2:
        raise ValueError("%s must be an int or a pair, got %r" % (name, v))
    return v


def _geom(inShape, wShape, stride, padding, dilation, groups):
    if len(inShape) != 5:
        raise RuntimeError("expected a 5 dimensional (N,C,H,W,T) tensor, got %d dimensions" % len(inShape))
    if len(wShape) == 5:
        if wShape[4] != 1:
            raise RuntimeError("the synapse kernel must have a time extent of 1, got %d" % wShape[4])
        wShape = wShape[:4]
    if len(wShape) != 4:
        raise RuntimeError("expected a weight of shape (O, C/groups, KH, KW[, 1]), got %r" % (tuple(wShape),))
    N, C, H, W, T = (int(v) for v in inShape)
    O, Cg, KH, KW = (int(v) for v in wShape)
    groups = int(groups)
    if groups < 1 or C % groups or O % groups or Cg * groups != C:
        raise RuntimeError("weight of shape %r does not fit %d input channels in %d groups"
                           % (tuple(wShape), C, groups))
    (sH, sW), (pH, pW), (dH, dW) = _pair(stride, "stride"), _pair(padding, "padding"), _pair(dilation, "dilation")
    return _lib.SynapseGeom(N, C, H, W, T, O, KH, KW, sH, sW, pH, pW, dH, dW, groups)


class _Plan:
    """What follows from the sizes of a layer alone: the geometry as the library takes it, its verdict, the shape of the
    output and the bytes of the weight gradient's workspace."""
    __slots__ = ("geom", "status", "outShape", "workspaceBytes")

    def __init__(self, *sizes):
        lib = _lib.load()
        self.geom = _geom(*sizes)
        OH, OW = ctypes.c_int32(), ctypes.c_int32()
        self.status = lib.slayer_synapse_out_shape(ctypes.byref(self.geom), ctypes.byref(OH), ctypes.byref(OW))
        self.outShape = (self.geom.N, self.geom.O, OH.value, OW.value, self.geom.T)
        self.workspaceBytes = lib.slayer_synapse_conv_grad_weight_workspace_bytes(ctypes.byref(self.geom))

    def checked(self):
        _lib.check(self.status, "slayer_synapse_out_shape")
        return self


# A training step of the convolutional network asks for 29 plans of 5 layers: 280 us of its 1440 us on the host when each was
# worked out anew.  (Kept by sizes, which determine them; the least recently used of 512 goes first.)
_keptPlan = functools.lru_cache(maxsize=512)(_Plan)


def _plan(inShape, wShape, stride, padding, dilation, groups):
    # whole numbers and tuples of them only: anything else is worked out (or refused) as it comes
    kinds = {type(groups)}
    for v in (inShape, wShape, stride, padding, dilation):
        if type(v) is not int:
            if not isinstance(v, tuple):
                return _Plan(inShape, wShape, stride, padding, dilation, groups)
            kinds.update(map(type, v))
    return (_keptPlan if kinds == {int} else _Plan)(inShape, wShape, stride, padding, dilation, groups)


def outShape(inShape, wShape, stride=1, padding=0, dilation=1, groups=1):
    """Shape (N, O, OH, OW, T) of ``conv`` for an input of shape ``inShape``."""
    return _plan(inShape, wShape, stride, padding, dilation, groups).checked().outShape


def supported(inShape, wShape, stride=1, padding=0, dilation=1, groups=1):
    """Whether the synapse kernels index this geometry: one batch item of the input and of the output below
    2 GiB, and a filter window - (padH + dilH * KH) rows plus (padW + dilW * KW) columns of the input - below
    16 MiB.  Decided on the host from the sizes alone (no GPU involved).  Beyond these limits the differentiable
    ``synapseConv`` / ``synapseConvTranspose`` fall back to torch's conv3d / conv_transpose3d, which the
    reference calls for every geometry."""
    plan = _plan(inShape, wShape, stride, padding, dilation, groups)
    return plan.status != 2 and plan.checked() is plan


def _triple(v, last):
    a, b = _pair(v, "argument")
    return (a, b, last)


def conv(input, weight, stride=1, padding=0, dilation=1, groups=1):
    """``F.conv3d(input, weight, None, (sH,sW,1), (pH,pW,0), (dH,dW,1), groups)`` for a weight of
    time extent 1."""
    out = host.conv2d(input, weight, stride, padding, dilation, groups)
    if out is not None:
        return out
    _check_input(input, "input")
    _check_input(weight, "weight")
    _check_device(input, weight, "input", "weight")
    plan = _plan(input.shape, weight.shape, stride, padding, dilation, groups).checked()
    g = plan.geom
    lib = _lib.load()
    out = torch.empty(plan.outShape, dtype=input.dtype, device=input.device)
    with _on_device_of(input) as stream:
        _lib.check(lib.slayer_synapse_conv_f32(_ptr(out), _ptr(input), _ptr(weight), ctypes.byref(g), stream),
                   "slayer_synapse_conv_f32")
    return out


def convGradInput(gradOutput, weight, inShape, stride=1, padding=0, dilation=1, groups=1):
    """Gradient of ``conv`` with respect to its input of shape ``inShape`` (= the transposed
    convolution of ``gradOutput``)."""
    _check_input(gradOutput, "gradOutput")
    _check_input(weight, "weight")
    _check_device(gradOutput, weight, "gradOutput", "weight")
    plan = _plan(inShape, weight.shape, stride, padding, dilation, groups).checked()
    g, expected = plan.geom, plan.outShape
    if tuple(gradOutput.shape) != expected:
        raise RuntimeError("gradOutput has shape %r, expected %r" % (tuple(gradOutput.shape), expected))
    lib = _lib.load()
    gradIn = torch.empty(tuple(int(v) for v in inShape), dtype=gradOutput.dtype, device=gradOutput.device)
    with _on_device_of(gradOutput) as stream:
        _lib.check(lib.slayer_synapse_conv_grad_input_f32(_ptr(gradIn), _ptr(gradOutput), _ptr(weight),
                                                          ctypes.byref(g), stream),
                   "slayer_synapse_conv_grad_input_f32")
    return gradIn


def convGradWeight(gradOutput, input, wShape, stride=1, padding=0, dilation=1, groups=1):
    """Gradient of ``conv`` with respect to its weight of shape ``wShape``."""
    _check_input(gradOutput, "gradOutput")
    _check_input(input, "input")
    _check_device(gradOutput, input, "gradOutput", "input")
    plan = _plan(input.shape, wShape, stride, padding, dilation, groups).checked()
    g, expected = plan.geom, plan.outShape
    if tuple(gradOutput.shape) != expected:
        raise RuntimeError("gradOutput has shape %r, expected %r" % (tuple(gradOutput.shape), expected))
    lib = _lib.load()
    gradW = torch.empty(tuple(int(v) for v in wShape), dtype=input.dtype, device=input.device)
    workspace = torch.empty((plan.workspaceBytes + 3) // 4, dtype=torch.float32, device=input.device)
    with _on_device_of(input) as stream:
        _lib.check(lib.slayer_synapse_conv_grad_weight_f32(_ptr(gradW), _ptr(gradOutput), _ptr(input),
                                                           _ptr(workspace), ctypes.byref(g), stream),
                   "slayer_synapse_conv_grad_weight_f32")
    return gradW


class _synapseConvFunction(Function):
    @staticmethod
    def forward(ctx, input, weight, stride, padding, dilation, groups):
        input = input.contiguous()
        weight = weight.contiguous()
        ctx.save_for_backward(input, weight)
        ctx.args = (stride, padding, dilation, groups)
        return conv(input, weight, *ctx.args)

    @staticmethod
    def backward(ctx, gradOutput):
        input, weight = ctx.saved_tensors
        gradOutput = gradOutput.contiguous()
        gradInput = gradWeight = None
        if ctx.needs_input_grad[0]:
            gradInput = host.conv2dGradInput(gradOutput, weight, input, *ctx.args)
            if gradInput is None:
                gradInput = convGradInput(gradOutput, weight, input.shape, *ctx.args)
        if ctx.needs_input_grad[1]:
            gradWeight = host.conv2dGradWeight(gradOutput, input, weight, *ctx.args)
            if gradWeight is None:
                gradWeight = convGradWeight(gradOutput, input, weight.shape, *ctx.args)
        return gradInput, gradWeight, None, None, None, None


class _synapseConvTransposeFunction(Function):
    """The transposed synapse: its forward pass is the input gradient of the convolution whose
    weight tensor it shares, its input gradient is that convolution."""

    @staticmethod
    def forward(ctx, input, weight, stride, padding, dilation, groups):
        input = input.contiguous()
        weight = weight.contiguous()
        (sH, sW), (pH, pW), (dH, dW) = _pair(stride, "stride"), _pair(padding, "padding"), _pair(dilation, "dilation")
        N, Cin, H, W, T = input.shape
        if weight.shape[0] != Cin:
            raise RuntimeError("weight of shape %r does not fit %d input channels" % (tuple(weight.shape), Cin))
        KH, KW = int(weight.shape[2]), int(weight.shape[3])
        outH = (H - 1) * sH - 2 * pH + dH * (KH - 1) + 1
        outW = (W - 1) * sW - 2 * pW + dW * (KW - 1) + 1
        ctx.outShape = (N, int(weight.shape[1]) * groups, outH, outW, T)
        ctx.save_for_backward(input, weight)
        ctx.args = (stride, padding, dilation, groups)
        return convGradInput(input, weight, ctx.outShape, *ctx.args)

    @staticmethod
    def backward(ctx, gradOutput):
        input, weight = ctx.saved_tensors
        gradOutput = gradOutput.contiguous()
        gradInput = gradWeight = None
        if ctx.needs_input_grad[0]:
            gradInput = conv(gradOutput, weight, *ctx.args)
        if ctx.needs_input_grad[1]:
            gradWeight = convGradWeight(input, gradOutput, weight.shape, *ctx.args)
        return gradInput, gradWeight, None, None, None, None


def synapseConv(input, weight, stride=1, padding=0, dilation=1, groups=1):
    """Differentiable ``conv``: stands where the reference calls ``F.conv3d(input, weight, None,
    stride, padding, dilation, groups)`` (src/slayer.py:499-507)."""
    if not supported(input.shape, weight.shape, stride, padding, dilation, groups):
        w5 = weight if weight.dim() == 5 else weight.unsqueeze(-1)
        return torch.nn.functional.conv3d(input, w5, None, _triple(stride, 1), _triple(padding, 0), _triple(dilation, 1),
                                          groups)
    return _synapseConvFunction.apply(input, weight, stride, padding, dilation, groups)


def synapseConvTranspose(input, weight, stride=1, padding=0, dilation=1, groups=1):
    """Differentiable transposed synapse: stands where the reference calls
    ``F.conv_transpose3d(input, weight, None, stride, padding, 0, groups, dilation)``
    (src/slayer.py:631-643)."""
    (sH, sW), (pH, pW), (dH, dW) = _pair(stride, "stride"), _pair(padding, "padding"), _pair(dilation, "dilation")
    KH, KW = int(weight.shape[2]), int(weight.shape[3])
    N, Cin, H, W, T = (int(v) for v in input.shape)
    # (the geometry of the convolution that this transposes: its input is this op's output)
    conv_in = (N, int(weight.shape[1]) * groups, (H - 1) * sH - 2 * pH + dH * (KH - 1) + 1,
               (W - 1) * sW - 2 * pW + dW * (KW - 1) + 1, T)
    if min(conv_in) >= 0 and not supported(conv_in, weight.shape[:4], stride, padding, dilation, groups):
        w5 = weight if weight.dim() == 5 else weight.unsqueeze(-1)
        return torch.nn.functional.conv_transpose3d(input, w5, None, _triple(stride, 1), _triple(padding, 0), 0, groups,
                                                    _triple(dilation, 1))
    return _synapseConvTransposeFunction.apply(input, weight, stride, padding, dilation, groups)


def _windows(inShape, wShape):
    """Extents of the pooled image: an extent that is no multiple of the window counts as extended by
    ``extent % window`` (src/slayer.py:565-575)."""
    H, W, KH, KW = int(inShape[2]), int(inShape[3]), int(wShape[2]), int(wShape[3])
    return (H + H % KH) // KH, (W + W % KW) // KW


def _check_window(weight):
    _check_input(weight, "weight")
    if weight.dim() not in (4, 5) or weight.numel() != weight.shape[2] * weight.shape[3]:
        raise RuntimeError("pooling takes a weight of shape (1, 1, KH, KW[, 1]), got %r" % (tuple(weight.shape),))


def pool(input, weight):
    """Sums over windows of ``weight``'s extent that do not overlap, channel by channel: ``conv`` with the window as
    stride on every channel by itself, ``input`` (N, C, H, W, T), ``weight`` (1, 1, KH, KW[, 1]).  ``None`` for sizes
    that the kernel does not take (:func:`poolSupported`)."""
    out = host.pool(input, weight)
    if out is not None:
        return out
    _check_input(input, "input")
    _check_window(weight)
    _check_device(input, weight, "input", "weight")
    if input.dim() != 5:
        raise RuntimeError("expected a 5 dimensional (N,C,H,W,T) tensor, got %d dimensions" % input.dim())
    N, C, H, W, T = input.shape
    lib = _lib.load()
    out = torch.empty((N, C) + _windows(input.shape, weight.shape) + (T,), dtype=input.dtype, device=input.device)
    with _on_device_of(input) as stream:
        status = lib.slayer_pool_f32(_ptr(out), _ptr(input), _ptr(weight), N, C, H, W, T, weight.shape[2], weight.shape[3],
                                     stream)
    if status == 2:
        return None
    _lib.check(status, "slayer_pool_f32")
    return out


def poolGradInput(gradOutput, weight, inShape, membranePotential=None, theta=0.0, tau=1.0, scale=1.0):
    """Gradient of :func:`pool` with respect to its input of shape ``inShape``; with a ``membranePotential`` of that shape
    times the surrogate gradient of ``slayerCuda.spikeBackward`` at it."""
    if membranePotential is not None and inShape == membranePotential.shape:
        out = host.poolSpikeBackward(gradOutput, weight, membranePotential, theta, tau, scale)
        if out is not None:
            return out
    _check_input(gradOutput, "gradOutput")
    _check_window(weight)
    _check_device(gradOutput, weight, "gradOutput", "weight")
    N, C, H, W, T = (int(v) for v in inShape)
    if tuple(gradOutput.shape) != (N, C) + _windows(inShape, weight.shape) + (T,):
        raise RuntimeError("gradOutput has shape %r, expected %r"
                           % (tuple(gradOutput.shape), (N, C) + _windows(inShape, weight.shape) + (T,)))
    if membranePotential is not None:
        _check_input(membranePotential, "membranePotential")
        _check_device(gradOutput, membranePotential, "gradOutput", "membranePotential")
        if tuple(membranePotential.shape) != (N, C, H, W, T):
            raise RuntimeError("membranePotential has shape %r, expected %r" % (tuple(membranePotential.shape), (N, C, H, W, T)))
    lib = _lib.load()
    gradIn = torch.empty((N, C, H, W, T), dtype=gradOutput.dtype, device=gradOutput.device)
    with _on_device_of(gradOutput) as stream:
        _lib.check(lib.slayer_pool_grad_input_f32(_ptr(gradIn), _ptr(gradOutput), _ptr(weight),
                                                  None if membranePotential is None else _ptr(membranePotential), theta, tau,
                                                  scale, N, C, H, W, T, weight.shape[2], weight.shape[3], stream),
                   "slayer_pool_grad_input_f32")
    return gradIn


def poolSpikeBackwardDelayedCorr(gradOutput, weight, membranePotential, filter, delaySteps, theta, tau, scale, Ts):
    """``slayerCuda.spikeBackwardDelayedCorr(poolGradInput(gradOutput, weight, membranePotential.shape), membranePotential,
    filter, delaySteps, ...)`` in one kernel, or ``None`` for rows and extents that it does not serve (nothing was launched);
    for shapes that :func:`poolSupported` takes."""
    for x, name in ((gradOutput, "gradOutput"), (membranePotential, "membranePotential"), (filter, "filter")):
        _check_input(x, name)
        _check_device(gradOutput, x, "gradOutput", name)
    _check_window(weight)
    _check_device(gradOutput, weight, "gradOutput", "weight")
    N, C, H, W, T = membranePotential.shape
    if tuple(gradOutput.shape) != (N, C) + _windows(membranePotential.shape, weight.shape) + (T,):
        raise RuntimeError("gradOutput has shape %r, which is not that of the pooled %r" % (tuple(gradOutput.shape), (N, C, H, W, T)))
    lib = _lib.load()
    gradIn = torch.empty_like(membranePotential)
    with _on_device_of(gradOutput) as stream:
        status = lib.slayer_pool_spike_bwd_delayed_corr_f32(
            _ptr(gradIn), _ptr(gradOutput), _ptr(weight), _ptr(membranePotential), _ptr(filter), N * C, H, W, T, weight.shape[2],
            weight.shape[3], filter.numel(), int(delaySteps), theta, tau, scale, Ts, stream)
    if status == 2:
        return None
    _lib.check(status, "slayer_pool_spike_bwd_delayed_corr_f32")
    return gradIn


class _synapsePoolFunction(Function):
    @staticmethod
    def forward(ctx, input, weight):
        ctx.save_for_backward(weight)
        ctx.inShape = tuple(input.shape)
        return pool(input, weight)

    @staticmethod
    def backward(ctx, gradOutput):
        (weight,) = ctx.saved_tensors
        return poolGradInput(gradOutput.contiguous(), weight, ctx.inShape), None


def poolSupported(inShape, wShape):
    """Whether the pooling kernels take these sizes: windows that lie in one channel each, on the image of a batch item's
    channels below one another (one channel, or an extended height that the window divides), at least one of them, and what
    the kernels index - one channel's image, and the image of all channels where the window divides the height, as in
    :func:`supported`."""
    N, C, H, W, T = (int(v) for v in inShape)
    KH, KW = int(wShape[2]), int(wShape[3])
    if min(_windows(inShape, wShape)) < 1 or (C > 1 and (H + H % KH) % KH != 0):
        return False
    limit = ((1 << 31) - (1 << 24)) // 4
    return (KH < 1024 and KW < 1024 and max(H, W) < (1 << 24) - 1024 and (H + KH) * (W + KW) * T < limit and N * C < (1 << 31)
            and (KH * W + KW) * T * 4 < (1 << 24) and N * C * ((H * W * ((T + 3) // 4)) // 256 + 1) < (1 << 31))


def synapsePool(input, weight):
    """Differentiable :func:`pool` for a weight that gets no gradient and sizes that :func:`poolSupported` takes."""
    return _synapsePoolFunction.apply(input.contiguous(), weight.contiguous())


def denseEventsSupported(N, K, O, T):
    """Whether ``denseEvents`` and ``denseEventsGradWeight`` take these extents (the limits the header states)."""
    lim = (1 << 31) - 64
    return N <= 65535 and N * O * T * 4 < lim and O <= 1024 and K * O * 4 < lim and 0 < K and N * T < (1 << 22) \
        and T < (1 << 21)


def denseEvents(input, weight):
    """``weight @ input[n]`` for every batch item, ``input`` (N, K, T), ``weight`` (O, K), summed over the
    non-zero inputs only (ascending k): the dense layer's product for spike tensors.  The work grows with
    the number of non-zero inputs."""
    out = host.denseEvents(input, weight)
    if out is not None:
        return out
    _check_input(input, "input")
    _check_input(weight, "weight")
    _check_device(input, weight, "input", "weight")
    if input.dim() != 3 or weight.dim() != 2 or weight.shape[1] != input.shape[1]:
        raise RuntimeError("denseEvents takes input (N, K, T) and weight (O, K); got %r and %r"
                           % (tuple(input.shape), tuple(weight.shape)))
    N, K, T = (int(v) for v in input.shape)
    O = int(weight.shape[0])
    lib = _lib.load()
    out = torch.empty((N, O, T), dtype=input.dtype, device=input.device)
    nbytes = lib.slayer_dense_events_workspace_bytes(N, K, O, T)
    workspace = torch.empty((nbytes + 3) // 4, dtype=torch.float32, device=input.device)
    with _on_device_of(input) as stream:
        _lib.check(lib.slayer_dense_events_f32(_ptr(out), _ptr(input), _ptr(weight), _ptr(workspace), N, K, O, T, stream),
                   "slayer_dense_events_f32")
    return out


def denseEventsGradWeight(gradOutput, input):
    """Weight gradient of the dense layer's product ``out[n] = weight @ input[n]``, ``input`` (N, K, T),
    ``gradOutput`` (N, O, T): ``sum_n gradOutput[n] @ input[n].T`` as (O, K), summed over the non-zero
    inputs only, in a fixed order.  The work grows with the number of non-zero inputs."""
    out = host.denseEventsGradWeight(gradOutput, input)
    if out is not None:
        return out
    _check_input(gradOutput, "gradOutput")
    _check_input(input, "input")
    _check_device(gradOutput, input, "gradOutput", "input")
    if input.dim() != 3 or gradOutput.dim() != 3 or gradOutput.shape[0] != input.shape[0] \
            or gradOutput.shape[2] != input.shape[2]:
        raise RuntimeError("denseEventsGradWeight takes gradOutput (N, O, T) and input (N, K, T); got %r and %r"
                           % (tuple(gradOutput.shape), tuple(input.shape)))
    N, K, T = (int(v) for v in input.shape)
    O = int(gradOutput.shape[1])
    lib = _lib.load()
    gradW = torch.empty((O, K), dtype=input.dtype, device=input.device)
    nbytes = lib.slayer_dense_events_grad_weight_workspace_bytes(N, K, O, T)
    workspace = torch.empty((nbytes + 3) // 4, dtype=torch.float32, device=input.device)
    with _on_device_of(input) as stream:
        _lib.check(lib.slayer_dense_events_grad_weight_f32(_ptr(gradW), _ptr(gradOutput), _ptr(input), _ptr(workspace),
                                                           N, K, O, T, stream),
                   "slayer_dense_events_grad_weight_f32")
    return gradW


def denseRowsSupported(N, K, O, T):
    """Whether ``denseRows`` takes these extents (the limits the header states)."""
    return bool(_lib.load().slayer_dense_rows_supported(N, K, O, T))


def denseRows(input, weight, transposed=False):
    """``weight @ input[n]`` for every batch item, ``input`` (N, K, T), ``weight`` (O, K) - or, ``transposed``,
    ``weight.T @ input[n]`` with ``weight`` (K, O): the dense layer's product and its input gradient on bf16
    matrix instructions over split operands (``slayer_dense_rows_f32``), for layers with up to a few hundred
    inputs."""
    _check_input(input, "input")
    _check_input(weight, "weight")
    _check_device(input, weight, "input", "weight")
    if input.dim() != 3 or weight.dim() != 2 or weight.shape[0 if transposed else 1] != input.shape[1]:
        raise RuntimeError("denseRows takes input (N, K, T) and weight (O, K), or (K, O) transposed; got %r and %r"
                           % (tuple(input.shape), tuple(weight.shape)))
    N, K, T = (int(v) for v in input.shape)
    O = int(weight.shape[1 if transposed else 0])
    lib = _lib.load()
    out = torch.empty((N, O, T), dtype=input.dtype, device=input.device)
    wRow, wCol = (1, O) if transposed else (K, 1)
    workspace = torch.empty((lib.slayer_dense_rows_workspace_bytes(K, O) + 3) // 4, dtype=torch.float32, device=input.device)
    with _on_device_of(input) as stream:
        _lib.check(lib.slayer_dense_rows_f32(_ptr(out), _ptr(weight), _ptr(input), _ptr(workspace), N, K, O, T, wRow, wCol,
                                             stream), "slayer_dense_rows_f32")
    return out


class _synapseDenseEventsFunction(Function):
    @staticmethod
    def forward(ctx, input, weight, product, gradient):
        ctx.save_for_backward(input, weight)
        ctx.gradient = gradient
        if product:
            return denseEvents(input, weight.contiguous())
        N, K, O = input.shape[0], input.shape[1], weight.shape[0]
        return torch.bmm(weight.unsqueeze(0).expand(N, O, K), input)

    @staticmethod
    def backward(ctx, gradOutput):
        input, weight = ctx.saved_tensors
        gradOutput = gradOutput.contiguous()
        gradInput = gradWeight = None
        if ctx.needs_input_grad[0]:   # the gradient is not sparse: a library product
            N, K, O = input.shape[0], input.shape[1], weight.shape[0]
            gradInput = torch.bmm(weight.t().unsqueeze(0).expand(N, K, O), gradOutput)
        if ctx.needs_input_grad[1]:
            if ctx.gradient:
                gradWeight = denseEventsGradWeight(gradOutput, input)
            else:
                gradWeight = torch.bmm(gradOutput, input.transpose(1, 2)).sum(0)
        return gradInput, gradWeight, None, None


def denseRowsGradWeightSupported(N, K, O, T):
    """Whether ``denseRowsGradWeight`` takes these extents (the limits the header states)."""
    return bool(_lib.load().slayer_dense_rows_grad_weight_supported(N, K, O, T))


def denseRowsGradWeight(gradOutput, input):
    """Weight gradient of the dense layer's product ``out[n] = weight @ input[n]``, ``input`` (N, K, T),
    ``gradOutput`` (N, O, T): ``sum_n gradOutput[n] @ input[n].T`` as (O, K), on bf16 matrix instructions over split
    operands (``slayer_dense_rows_grad_weight_f32``), for layers with up to 448 inputs and 256 outputs."""
    _check_input(gradOutput, "gradOutput")
    _check_input(input, "input")
    _check_device(gradOutput, input, "gradOutput", "input")
    if input.dim() != 3 or gradOutput.dim() != 3 or gradOutput.shape[0] != input.shape[0] \
            or gradOutput.shape[2] != input.shape[2]:
        raise RuntimeError("denseRowsGradWeight takes gradOutput (N, O, T) and input (N, K, T); got %r and %r"
                           % (tuple(gradOutput.shape), tuple(input.shape)))
    N, K, T = (int(v) for v in input.shape)
    O = int(gradOutput.shape[1])
    lib = _lib.load()
    gradW = torch.empty((O, K), dtype=input.dtype, device=input.device)
    nbytes = lib.slayer_dense_rows_grad_weight_workspace_bytes(N, K, O, T)
    workspace = torch.empty((nbytes + 3) // 4, dtype=torch.float32, device=input.device)
    with _on_device_of(input) as stream:
        _lib.check(lib.slayer_dense_rows_grad_weight_f32(_ptr(gradW), _ptr(gradOutput), _ptr(input), _ptr(workspace),
                                                         N, K, O, T, stream), "slayer_dense_rows_grad_weight_f32")
    return gradW


DENSE_ROWS_MAX_INPUTS = 448   # two launches of slayer_dense_rows_f32; beyond that the library product


def denseRowsPays(N, K, O, T):
    """Whether the dense layer's product (N, K, T) -> (N, O, T) is taken by ``denseRows``: few enough inputs, and enough
    work for a kernel that keeps the weights in registers (a library product is as fast on small problems)."""
    return K <= DENSE_ROWS_MAX_INPUTS and N * T >= 2048 and O >= 16 and denseRowsSupported(N, K, O, T)


def _aligned(t):
    """``t`` contiguous and on a 16-byte boundary (a view that starts inside an allocation is copied)."""
    t = t.contiguous()
    return t if t.data_ptr() % 16 == 0 else t.clone()


class _synapseDenseRowsFunction(Function):
    @staticmethod
    def forward(ctx, input, weight):
        ctx.save_for_backward(input, weight)
        return denseRows(input, weight.contiguous())

    @staticmethod
    def backward(ctx, gradOutput):
        input, weight = ctx.saved_tensors
        gradOutput = _aligned(gradOutput)
        gradInput = gradWeight = None
        N, K, T = input.shape
        O = weight.shape[0]
        if ctx.needs_input_grad[0]:
            if denseRowsPays(N, O, K, T):     # (the outputs are what is summed over now)
                gradInput = denseRows(gradOutput, weight.contiguous(), transposed=True)
            else:
                gradInput = torch.bmm(weight.t().unsqueeze(0).expand(N, K, O), gradOutput)
        if ctx.needs_input_grad[1]:
            if N * T >= 2048 and denseRowsGradWeightSupported(N, K, O, T):
                gradWeight = denseRowsGradWeight(gradOutput, input)
            else:
                gradWeight = torch.bmm(gradOutput, input.transpose(1, 2)).sum(0)
        return gradInput, gradWeight


def _thin_extents(x, weight, channels):
    if x.dim() != 3 or weight.dim() != 2 or weight.shape[channels] != x.shape[1]:
        raise RuntimeError("the dense layer takes tensors (N, channels, T) and a weight (O, K); got %r and %r"
                           % (tuple(x.shape), tuple(weight.shape)))
    return x.shape[0], weight.shape[1], weight.shape[0], x.shape[2]


def _workspace(nbytes, like):
    return torch.empty((nbytes + 3) // 4, dtype=torch.float32, device=like.device) if nbytes else None


def denseThin(input, weight):
    """``weight @ input[n]`` for every batch item, ``input`` (N, K, T), ``weight`` (O, K), for few outputs
    (``slayer_dense_thin_f32``)."""
    out = host.denseThin(input, weight)
    if out is not None:
        return out
    _check_input(input, "input")
    _check_input(weight, "weight")
    _check_device(input, weight, "input", "weight")
    N, K, O, T = _thin_extents(input, weight, 1)
    lib = _lib.load()
    out = torch.empty((N, O, T), dtype=input.dtype, device=input.device)
    workspace = _workspace(lib.slayer_dense_thin_workspace_bytes(N, K, O, T, 0), input)
    with _on_device_of(input) as stream:
        _lib.check(lib.slayer_dense_thin_f32(_ptr(out), _ptr(weight), _ptr(input), None if workspace is None else _ptr(workspace),
                                             N, K, O, T, stream), "slayer_dense_thin_f32")
    return out


def denseThinGradInput(gradOutput, weight):
    """``weight.T @ gradOutput[n]`` for every batch item, ``gradOutput`` (N, O, T), ``weight`` (O, K)."""
    out = host.denseThinGradInput(gradOutput, weight)
    if out is not None:
        return out
    _check_input(gradOutput, "gradOutput")
    _check_input(weight, "weight")
    _check_device(gradOutput, weight, "gradOutput", "weight")
    N, K, O, T = _thin_extents(gradOutput, weight, 0)
    lib = _lib.load()
    gradIn = torch.empty((N, K, T), dtype=gradOutput.dtype, device=gradOutput.device)
    with _on_device_of(gradOutput) as stream:
        _lib.check(lib.slayer_dense_thin_grad_input_f32(_ptr(gradIn), _ptr(weight), _ptr(gradOutput), N, K, O, T, stream),
                   "slayer_dense_thin_grad_input_f32")
    return gradIn


def denseThinGradWeight(gradOutput, input):
    """``sum_n gradOutput[n] @ input[n].T`` as (O, K), ``gradOutput`` (N, O, T), ``input`` (N, K, T)."""
    out = host.denseThinGradWeight(gradOutput, input)
    if out is not None:
        return out
    _check_input(gradOutput, "gradOutput")
    _check_input(input, "input")
    _check_device(gradOutput, input, "gradOutput", "input")
    if input.dim() != 3 or gradOutput.dim() != 3 or gradOutput.shape[0] != input.shape[0] \
            or gradOutput.shape[2] != input.shape[2]:
        raise RuntimeError("denseThinGradWeight takes gradOutput (N, O, T) and input (N, K, T); got %r and %r"
                           % (tuple(gradOutput.shape), tuple(input.shape)))
    N, K, T = input.shape
    O = gradOutput.shape[1]
    lib = _lib.load()
    gradW = torch.empty((O, K), dtype=input.dtype, device=input.device)
    workspace = _workspace(lib.slayer_dense_thin_workspace_bytes(N, K, O, T, 1), input)
    with _on_device_of(input) as stream:
        _lib.check(lib.slayer_dense_thin_grad_weight_f32(_ptr(gradW), _ptr(gradOutput), _ptr(input),
                                                         None if workspace is None else _ptr(workspace), N, K, O, T, stream),
                   "slayer_dense_thin_grad_weight_f32")
    return gradW


def denseThinPays(N, K, O, T):
    """Whether the layer's product (N, K, T) -> (N, O, T) is taken by the kernels for few outputs: up to 16, or up to 32 where
    the layer is so small that its launches count more than its work."""
    # (us on the GPU, the same tensors again and again, ours / library: 4096 -> 10 at (1, 300) 5.4 / 14, (12, 300) 16 / 24,
    # (64, 300) 66 / 82, (256, 300) 250 / 228; 5760 -> 10 at (5, 173) 9.4 / 22; 512 -> 10 at (1, 350) 3.8 / 5.5, (12, 350) 5.9 /
    # 8.2; 256 -> 8 at (64, 2000) 24 / 25; 2048 -> 16 at (64, 300) 34 / 40; 1024 -> 16 at (128, 1000) 105 / 93.  Input gradient: 4096 -> 10 at (12, 300) 13 / 32, (64, 300) 65 / 130;
    # 512 -> 10 at (12, 350) 5.1 / 12; 512 -> 11 at (4, 1450) 5.6 / 9.0; 256 -> 8 at (64, 2000) 23 / 57.  Weight gradient: 4096 ->
    # 10 at (12, 300) 19 / 27, (64, 300) 64 / 94; 512 -> 10 at (1, 350) 5.6 / 7.6, (12, 350) 8.3 / 12; 2048 -> 16 at (64, 300)
    # 45 / 40.  More than 16 outputs, product; input gradient; weight gradient: 250 -> 25 at (1, 500) 3.7 / 5.7; 4.5 / 4.2; 5.4 /
    # 25; 512 -> 32 at (4, 500) 5.0 / 6.5; 5.8 / 5.6; 7.9 / 8.4; 1024 -> 17 at (1, 300) 6.0 / 7.2; 4.6 / 4.6; 5.4 / 7.6; 4096 -> 32
    # at (1, 250) 6.4 / 24; 5.5 / 6.0; 5.5 / 8.5; 300 -> 20 at (1, 37) 3.8 / 6.9; 4.8 / 4.1; 4.2 / 6.7: of 27 such sizes up to the
    # limit none is slower in all three together.  On the host a product of the library's and its gradients take 90 us, these 30.)
    return (O <= 16 or (O <= 32 and N * K * T <= 1 << 20)) and bool(_lib.load().slayer_dense_thin_supported(N, K, O, T))


def plainTensors(*tensors):
    """Whether nothing but autograd looks at operations on these tensors: no transform, no forward-mode derivative, no
    tracing or compiling, no autocast, no mode and no subclass that an autograd Function would hide the operation from."""
    return (host.unwrapped(*tensors)
            and not torch._C._are_functorch_transforms_active() and torch.autograd.forward_ad._current_level < 0
            and torch._C._len_torch_dispatch_stack() == 0 and torch._C._len_torch_function_stack() == 0
            and not torch.is_autocast_enabled("cuda") and torch._C._get_tracing_state() is None
            and not torch.compiler.is_compiling())


class _synapseDenseThinFunction(Function):
    """The product and its gradients for few outputs.  A backward pass that is itself recorded (``create_graph``), or whose
    gradients are not plain tensors (``is_grads_batched``), is torch's."""

    @staticmethod
    def forward(ctx, input, weight):
        ctx.save_for_backward(input, weight)
        return denseThin(input, weight.contiguous())

    @staticmethod
    def backward(ctx, gradOutput):
        input, weight = ctx.saved_tensors
        gradInput = gradWeight = None
        N, K, T = input.shape
        O = weight.shape[0]
        # (of what plainTensors looks for, what can be there in a backward pass)
        own = not torch.is_grad_enabled() and gradOutput.dtype == torch.float32 and host.unwrapped(gradOutput, input, weight) \
            and torch.autograd.forward_ad._current_level < 0 and torch._C._len_torch_dispatch_stack() == 0
        if own:
            gradOutput = gradOutput.contiguous()
        if ctx.needs_input_grad[0]:
            if own:
                gradInput = denseThinGradInput(gradOutput, weight.contiguous())
            else:
                gradInput = torch.bmm(weight.t().unsqueeze(0).expand(N, K, O), gradOutput)
        if ctx.needs_input_grad[1]:
            if own:
                gradWeight = denseThinGradWeight(gradOutput, input.contiguous())
            else:
                gradWeight = torch.bmm(gradOutput, input.transpose(1, 2)).sum(0)
        return gradInput, gradWeight


def synapseDenseThin(input, weight):
    """``weight @ input[n]`` for every batch item (``input`` (N, K, T), ``weight`` (O, K)) with its gradients, for layers with
    few outputs (:func:`denseThinPays`)."""
    return _synapseDenseThinFunction.apply(input.contiguous(), weight)


def synapseDenseRows(input, weight):
    """``weight @ input[n]`` for every batch item (``input`` (N, K, T), ``weight`` (O, K)) with its gradients, for
    layers with few inputs: product and input gradient from ``denseRows`` (bf16 matrix instructions over split
    operands, weights in registers), the weight gradient from ``denseRowsGradWeight`` (the library's batched product
    for more than 448 inputs or 256 outputs)."""
    return _synapseDenseRowsFunction.apply(_aligned(input), weight)


def synapseDenseEvents(input, weight, product=True, gradient=True):
    """``weight @ input[n]`` for every batch item (``input`` (N, K, T), ``weight`` (O, K)) with its gradients,
    for inputs that are spike tensors: the product (``product``) and the weight gradient (``gradient``) summed
    over the non-zero inputs (``denseEvents``, ``denseEventsGradWeight``) or as library matrix products; the
    input gradient - a product with the dense output gradient - always from the library."""
    return _synapseDenseEventsFunction.apply(input.contiguous(), weight, product, gradient)
