"""Convolution layers of the MaterialGAN caller's networks on the matrix-core
kernels of libsvbrdf_hip.so (csrc/conv.hip, conv_split.hip, generator.hip).

* :func:`conv3x3` -- a 3x3 convolution (stride 1, zero padding 1) with the
  fused epilogue of the reference's blocks: ``act(conv + noise_strength *
  noise + bias)``, act = identity, ReLU (VGG, src/descriptor.py:7-79) or
  leaky ReLU x sqrt(2) (ModulateConvBlock,
  src/higan_models/stylegan2_generator_network.py:738-755).  Differentiable
  with respect to the input, the weights and the noise map: the forward and
  dL/dx are the HIP kernel (dL/dx is the convolution of dL/dy with the
  flipped, transposed weights; where only dL/dx is wanted the kernel applies
  the activation's derivative to dL/dy itself, :func:`conv3x3_input_grad`),
  and so is dL/dweights (:func:`conv3x3_wgrad`, an MFMA GEMM over the pixels
  with the nine taps sharing the dL/dy operand).
* :func:`upsample2` -- x2 upsampling by zero insertion and the [1, 3, 3, 1]
  filter (UpsamplingLayer, stylegan2_generator_network.py:419-479); forward
  and adjoint are HIP kernels.
* :class:`Conv3x3` -- a frozen 3x3 layer (VGG): weights packed once, in both
  layouts; outside autograd it can write a second, scaled copy of its output.
* :func:`modulated_conv3x3`, :class:`StyleLayersFunction`,
  :class:`ToRGBFunction` -- a StyleGAN2 block's convolution, every layer's
  style in one launch, and the output layer with its skip image.
"""
import numpy as np
import torch

from . import _lib

ACT = {"none": _lib.ACT_NONE, "relu": _lib.ACT_RELU, "lrelu": _lib.ACT_LRELU}


def plain(module, kind):
    """Whether calling module is kind.forward and nothing else: no subclass or
    replacement of it and no hooks.  What passes a module's call by asks first."""
    return (type(module) is kind and "forward" not in module.__dict__
            and not (module._forward_hooks or module._forward_pre_hooks or module._backward_hooks
                     or module._backward_pre_hooks)
            and not torch.nn.modules.module._has_any_global_hook())


def _check(t, name):
    if t.device.type != "cuda" or t.dtype != torch.float32:
        raise ValueError(f"{name} must be a float32 CUDA tensor (there is no CPU path), got {t.dtype} on {t.device}")


def _pack_inputs(weight, style):
    w = weight.detach().contiguous()
    _check(w, "weight")
    if tuple(w.shape[2:]) != (3, 3):
        raise ValueError(f"weight must be [Cout, Cin, 3, 3], got {tuple(w.shape)}")
    st = None
    if style is not None:
        st = style.detach().reshape(-1).contiguous()
        _check(st, "style")
        if st.numel() != int(w.shape[1]):
            raise ValueError(f"style must have {int(w.shape[1])} values, got {st.numel()}")
    return w, st


def pack3x3(weight, style=None, scale=1.0, demodulate=False, transpose=False):
    """[Cout, Cin, 3, 3] -> the kernel's layout ([9, Cin, Cout], or the input-
    gradient layout [9, Cout, Cin] with flipped taps when transpose), times
    scale * style[ci] and demodulated per output channel when asked."""
    w, st = _pack_inputs(weight, style)
    cout, cin = int(w.shape[0]), int(w.shape[1])
    out = torch.empty((9, cout, cin) if transpose else (9, cin, cout), dtype=torch.float32, device=w.device)
    _lib.call("svbrdf_conv3x3_pack", _lib.ptr(w), cout, cin, _lib.ptr(st), float(scale), int(bool(demodulate)),
              int(bool(transpose)), _lib.ptr(out), _lib.stream_handle(w.device))
    return out


def _takes_split(n, cin, h, w, cout, from_packed=False):
    """Whether a shape runs on the bf16 matrix cores with split operands
    (fp32 results; csrc/conv_split.hip); from_packed: where this call has to
    split packed weights first."""
    rule = "svbrdf_conv3x3_split_packed_preferred" if from_packed else "svbrdf_conv3x3_split_preferred"
    return bool(_lib.query(rule, n, cin, h, w, cout))


def _split_buffer(cin, cout, device):
    return torch.empty(int(_lib.query("svbrdf_conv3x3_split_weights_bytes", cin, cout)) // 4, dtype=torch.float32,
                       device=device)


def _version(t):
    """Counts the writes to a tensor (None in inference mode, which has no count)."""
    return None if t.is_inference() else t._version


def _split_packed(packed):
    """Split weights of a convolution from its packed ones ([9, Cin, Cout])."""
    _, cin, cout = (int(s) for s in packed.shape)
    packed = packed.contiguous()
    out = _split_buffer(cin, cout, packed.device)
    _lib.call("svbrdf_conv3x3_split_packed", _lib.ptr(packed), cin, cout, _lib.ptr(out),
              _lib.stream_handle(packed.device))
    return out


def _pack_for(n, h, w, weight, style=None, scale=1.0, demodulate=False, transpose=False):
    """(packed, split) weights for a convolution of n images of h x w: the
    layout that its path reads, the other None."""
    cout, cin = int(weight.shape[0]), int(weight.shape[1])
    k, m = (cout, cin) if transpose else (cin, cout)
    if not _takes_split(n, k, h, w, m):
        return pack3x3(weight, style, scale, demodulate, transpose), None
    wt, st = _pack_inputs(weight, style)
    out = _split_buffer(k, m, wt.device)
    _lib.call("svbrdf_conv3x3_pack_split", _lib.ptr(wt), cout, cin, _lib.ptr(st), float(scale), int(bool(demodulate)),
              int(bool(transpose)), _lib.ptr(out), _lib.stream_handle(wt.device))
    return None, out


def conv3x3_packed(x, packed, cout, bias=None, noise=None, noise_strength=0.0, act="none"):
    """The kernel itself on packed weights: x [N, Cin, H, W] -> [N, Cout, H, W]."""
    x = x.contiguous()
    _check(x, "x")
    n, cin, h, w = (int(s) for s in x.shape)
    if tuple(packed.shape) != (9, cin, cout):
        raise ValueError(f"packed weights {tuple(packed.shape)} do not match Cin={cin}, Cout={cout}")
    split = _split_packed(packed) if _takes_split(n, cin, h, w, cout, from_packed=True) else None
    return _conv3x3(x, packed, split, cin, cout, bias, noise, noise_strength, act)


def _check_tap(tap, x, size):
    _check(tap, "tap")
    if tap.numel() != size or tap.device != x.device or not tap.is_contiguous():
        raise ValueError(f"tap must hold {size} contiguous values on {x.device}, got {tap.numel()} on {tap.device}")


def _conv_inputs(x, bias, noise):
    """A convolution's input, bias and noise as the kernels read them."""
    x = x.contiguous()
    _check(x, "x")
    if bias is not None:
        bias = bias.detach().reshape(-1).contiguous()
        _check(bias, "bias")
    if noise is not None:
        noise = noise.detach().reshape(-1).contiguous()
        _check(noise, "noise")
        if noise.numel() != x.shape[2] * x.shape[3]:
            raise ValueError(f"noise must have {x.shape[2] * x.shape[3]} values, got {noise.numel()}")
    return x, bias, noise


def _conv3x3(x, packed, split, cin, cout, bias=None, noise=None, noise_strength=0.0, act="none", tap=None,
             tap_scale=1.0):
    """conv3x3_packed on the split weights, or on the packed ones where those
    are None; cin, cout: the weights'.  tap: a flat tensor of the output's
    size that receives tap_scale times it."""
    n, channels, h, w = (int(s) for s in x.shape)
    if channels != cin:
        raise ValueError(f"x has {channels} channels, the weights Cin={cin}")
    x, bias, noise = _conv_inputs(x, bias, noise)
    y = torch.empty((n, cout, h, w), dtype=torch.float32, device=x.device)
    # K-split partial sums of small images (torch's caching allocator makes
    # this a free-list lookup after the first call)
    kind = "svbrdf_conv3x3" if split is None else "svbrdf_conv3x3_split"
    ws_bytes = int(_lib.query(f"{kind}_workspace_bytes", n, cin, h, w, cout))
    ws = torch.empty(ws_bytes // 4, dtype=torch.float32, device=x.device) if ws_bytes else None
    if tap is not None:
        _check_tap(tap, x, y.numel())
        _lib.call("svbrdf_conv3x3_tapped", _lib.ptr(x), n, cin, h, w, _lib.ptr(packed), _lib.ptr(split), cout,
                  _lib.ptr(bias), _lib.ptr(noise), float(noise_strength), ACT[act], _lib.ptr(y), _lib.ptr(tap),
                  float(tap_scale), _lib.ptr(ws), ws_bytes, _lib.stream_handle(x.device))
        return y
    _lib.call(kind, _lib.ptr(x), n, cin, h, w, _lib.ptr(packed if split is None else split), cout, _lib.ptr(bias),
              _lib.ptr(noise), float(noise_strength), ACT[act], _lib.ptr(y), _lib.ptr(ws), ws_bytes,
              _lib.stream_handle(x.device))
    return y


def conv3x3_input_grad(grad_y, y, packed_t, cin, act):
    """dL/dx of y = act(conv3x3(x, w) + ...) from dL/dy and y, with the
    flipped, transposed weights of pack3x3(w, transpose=True): the kernel
    gates dL/dy by the activation's derivative while it stages it."""
    g = grad_y.contiguous()
    _check(g, "grad_y")
    y = y.contiguous()
    _check(y, "y")
    n, cout, h, w = (int(s) for s in g.shape)
    if tuple(y.shape) != tuple(g.shape):
        raise ValueError(f"y {tuple(y.shape)} and grad_y {tuple(g.shape)} differ")
    if tuple(packed_t.shape) != (9, cout, cin):
        raise ValueError(f"packed weights {tuple(packed_t.shape)} do not match Cout={cout}, Cin={cin}")
    split_t = _split_packed(packed_t) if _takes_split(n, cout, h, w, cin, from_packed=True) else None
    return _input_grad(g, y, packed_t, split_t, cin, act)


def _input_grad(grad_y, y, packed_t, split_t, cin, act):
    """conv3x3_input_grad on the split weights, or on the packed ones where those are None."""
    g, y = grad_y.contiguous(), y.contiguous()
    _check(g, "grad_y")
    _check(y, "y")
    n, cout, h, w = (int(s) for s in g.shape)
    gx = torch.empty((n, cin, h, w), dtype=torch.float32, device=g.device)
    kind = "" if split_t is None else "_split"
    ws_bytes = int(_lib.query(f"svbrdf_conv3x3{kind}_workspace_bytes", n, cout, h, w, cin))
    ws = torch.empty(ws_bytes // 4, dtype=torch.float32, device=g.device) if ws_bytes else None
    _lib.call(f"svbrdf_conv3x3_input_grad{kind}", _lib.ptr(g), _lib.ptr(y), ACT[act], n, cout, h, w,
              _lib.ptr(packed_t if split_t is None else split_t), cin, _lib.ptr(gx), _lib.ptr(ws), ws_bytes,
              _lib.stream_handle(g.device))
    return gx


def conv3x3_wgrad(x, grad_z, cout):
    """dL/dw [cout, Cin, 3, 3] of a 3x3 convolution (padding 1) from its input
    x [N, Cin, H, W] and grad_z [N, cout, H, W], the gradient with respect to
    its output before bias and activation (torch.nn.grad.conv2d_weight)."""
    x = x.contiguous()
    g = grad_z.contiguous()
    _check(x, "x")
    _check(g, "grad_z")
    n, cin, h, w = (int(s) for s in x.shape)
    if tuple(g.shape) != (n, cout, h, w):
        raise ValueError(f"grad_z {tuple(g.shape)} does not match x {tuple(x.shape)} and Cout={cout}")
    gw = torch.empty((cout, cin, 3, 3), dtype=torch.float32, device=x.device)
    ws_bytes = int(_lib.query("svbrdf_conv3x3_wgrad_workspace_bytes", n, cin, h, w, cout))
    ws = torch.empty(ws_bytes // 4, dtype=torch.float32, device=x.device) if ws_bytes else None
    _lib.call("svbrdf_conv3x3_wgrad", _lib.ptr(x), _lib.ptr(g), n, cin, h, w, cout, _lib.ptr(gw), _lib.ptr(ws),
              ws_bytes, _lib.stream_handle(x.device))
    return gw


_ACT_SLOPES = {"relu": (1.0, 0.0), "lrelu": (1.4142135623730951, 0.2 * 1.4142135623730951)}


def _act_grad(grad_y, y, act):
    """dL/d(pre-activation) from dL/dy and y (the activations keep the sign):
    one HIP kernel, grad_y * (y > 0 ? pos : neg)."""
    if act not in _ACT_SLOPES:
        return grad_y
    g, yy = grad_y.contiguous(), y.contiguous()
    out = torch.empty_like(g)
    pos, neg = _ACT_SLOPES[act]
    _lib.call("svbrdf_act_grad", _lib.ptr(g), _lib.ptr(yy), g.numel(), pos, neg, _lib.ptr(out),
              _lib.stream_handle(g.device))
    return out


class Conv3x3Function(torch.autograd.Function):
    """y = act(conv3x3(x, weight) + noise_strength * noise + bias)."""

    @staticmethod
    def forward(ctx, x, weight, bias, noise, noise_strength, act):
        n, _, h, w = x.shape
        cout, cin = (int(s) for s in weight.shape[:2])
        y = _conv3x3(x, *_pack_for(n, h, w, weight), cin, cout, bias, noise, noise_strength, act)
        ctx.save_for_backward(x, weight, noise, y)
        ctx.noise_strength, ctx.act = float(noise_strength), act
        return y

    @staticmethod
    def backward(ctx, grad_y):
        x, weight, noise, y = ctx.saved_tensors
        gx = gw = gnoise = None
        need_gz = ctx.needs_input_grad[1] or (ctx.needs_input_grad[3] and noise is not None)
        if not need_gz:
            # only dL/dx: the gate is applied inside the convolution
            if ctx.needs_input_grad[0]:
                n, _, h, w = y.shape
                gx = _input_grad(grad_y, y, *_pack_for(n, h, w, weight, transpose=True), int(weight.shape[1]), ctx.act)
            return gx, None, None, None, None, None
        gz = _act_grad(grad_y.contiguous(), y, ctx.act).contiguous()
        if ctx.needs_input_grad[0]:
            n, _, h, w = y.shape
            gx = _conv3x3(gz, *_pack_for(n, h, w, weight, transpose=True), int(weight.shape[0]), int(weight.shape[1]))
        if ctx.needs_input_grad[1]:
            gw = conv3x3_wgrad(x, gz, int(weight.shape[0]))
        if ctx.needs_input_grad[3] and noise is not None:
            gnoise = (ctx.noise_strength * gz.sum(dim=(0, 1))).reshape(noise.shape)
        return gx, gw, None, gnoise, None, None


def conv3x3(x, weight, bias=None, noise=None, noise_strength=0.0, act="none"):
    if act not in ACT:
        raise ValueError(f"act must be one of {sorted(ACT)}")
    return Conv3x3Function.apply(x, weight, bias, noise, noise_strength, act)


def modulation_grad(weight, style, scale, demodulate, grad_weight):
    """dL/dstyle [Cin] of the weights pack3x3(weight, style, scale,
    demodulate) packs, from dL/d(those weights) in [Cout, Cin, 3, 3]."""
    w = weight.detach().contiguous()
    g = grad_weight.contiguous()
    st = style.detach().reshape(-1).contiguous()
    for t, name in ((w, "weight"), (g, "grad_weight"), (st, "style")):
        _check(t, name)
    cout, cin = int(w.shape[0]), int(w.shape[1])
    if tuple(g.shape) != tuple(w.shape) or st.numel() != cin:
        raise ValueError(f"grad_weight {tuple(g.shape)} / style {st.numel()} do not match weight {tuple(w.shape)}")
    ws = torch.empty(2 * cout, dtype=torch.float32, device=w.device)
    out = torch.empty(cin, dtype=torch.float32, device=w.device)
    _lib.call("svbrdf_conv3x3_modulation_grad", _lib.ptr(w), cout, cin, _lib.ptr(st), float(scale),
              int(bool(demodulate)), _lib.ptr(g), _lib.ptr(out), _lib.ptr(ws), ws.numel() * 4,
              _lib.stream_handle(w.device))
    return out


def _small_modconv(x, weight, style, scale, demodulate, bias, noise, noise_strength, act):
    """A modulated convolution of a few pixels from the weights themselves;
    None for the shapes that pack them (svbrdf_modconv3x3_small takes one
    sample of at most 128 pixels, channels in eights, aligned weights)."""
    wt, st = _pack_inputs(weight, style)
    cout, cin = int(wt.shape[0]), int(wt.shape[1])
    n, channels, h, w = (int(s) for s in x.shape)
    if n != 1 or channels != cin or wt.data_ptr() % 16:
        return None
    ws_bytes = int(_lib.query("svbrdf_modconv3x3_small_workspace_bytes", cin, h, w, cout))
    if not ws_bytes:
        return None
    x, bias, noise = _conv_inputs(x, bias, noise)
    y = torch.empty((1, cout, h, w), dtype=torch.float32, device=x.device)
    ws = torch.empty(ws_bytes // 4, dtype=torch.float32, device=x.device)
    _lib.call("svbrdf_modconv3x3_small", _lib.ptr(x), cin, h, w, _lib.ptr(wt), cout, _lib.ptr(st), float(scale),
              int(bool(demodulate)), _lib.ptr(bias), _lib.ptr(noise), float(noise_strength), ACT[act], _lib.ptr(y),
              _lib.ptr(ws), ws_bytes, _lib.stream_handle(x.device))
    return y


class ModConv3x3Function(torch.autograd.Function):
    """The modulated 3x3 convolution of a StyleGAN2 block (batch 1):
    y = act(conv3x3(x, w') + noise_strength * noise + bias) with
    w'[co][ci] = scale style[ci] w[co][ci], divided per output channel by
    sqrt(sum w'^2 + 1e-8) when demodulate (ModulateConvBlock.forward,
    src/higan_models/stylegan2_generator_network.py:694-755).  The modulation
    and demodulation happen inside the weight packing; the backward gives
    dL/dx, dL/dstyle (through svbrdf_conv3x3_modulation_grad) and dL/dnoise.
    The base weight w is frozen (the caller optimises latents and noise)."""

    @staticmethod
    def forward(ctx, x, style, weight, scale, demodulate, bias, noise, noise_strength, act):
        if weight.requires_grad:
            raise ValueError("ModConv3x3Function keeps the base weight frozen; use conv3x3 with explicitly "
                             "modulated weights to train it")
        n, _, h, w = x.shape
        cout, cin = (int(s) for s in weight.shape[:2])
        y = _small_modconv(x, weight, style, scale, demodulate, bias, noise, noise_strength, act)
        if y is None:
            y = _conv3x3(x, *_pack_for(n, h, w, weight, style, scale, demodulate), cin, cout, bias, noise,
                         noise_strength, act)
        ctx.save_for_backward(x, style, weight, noise, y)
        ctx.scale, ctx.demodulate = float(scale), bool(demodulate)
        ctx.noise_strength, ctx.act = float(noise_strength), act
        return y

    @staticmethod
    def backward(ctx, grad_y):
        x, style, weight, noise, y = ctx.saved_tensors
        gx = gstyle = gnoise = None
        cin = int(weight.shape[1])
        need_gx, need_gs = ctx.needs_input_grad[0], ctx.needs_input_grad[1]
        need_gn = ctx.needs_input_grad[6] and noise is not None
        if need_gx:
            n, _, h, w = y.shape
            packed_t = _pack_for(n, h, w, weight, style, ctx.scale, ctx.demodulate, transpose=True)
        if not (need_gs or need_gn):
            if need_gx:
                gx = _input_grad(grad_y, y, *packed_t, cin, ctx.act)
            return gx, None, None, None, None, None, None, None, None
        gz = _act_grad(grad_y.contiguous(), y, ctx.act).contiguous()
        if need_gx:
            gx = _conv3x3(gz, *packed_t, int(weight.shape[0]), cin)
        if need_gs:
            gw = conv3x3_wgrad(x, gz, int(weight.shape[0]))
            gstyle = modulation_grad(weight, style, ctx.scale, ctx.demodulate, gw).reshape(style.shape)
        if need_gn:
            gnoise = (ctx.noise_strength * gz.sum(dim=(0, 1))).reshape(noise.shape)
        return gx, gstyle, None, None, None, None, gnoise, None, None


def modulated_conv3x3(x, style, weight, scale, demodulate=True, bias=None, noise=None, noise_strength=0.0,
                      act="none"):
    if act not in ACT:
        raise ValueError(f"act must be one of {sorted(ACT)}")
    if x.shape[0] != 1:
        raise ValueError("modulated_conv3x3 takes one sample (the style is per input channel)")
    return ModConv3x3Function.apply(x, style, weight, scale, demodulate, bias, noise, noise_strength, act)


MAX_RGB = 9   # output channels of svbrdf_torgb
_STYLE_LAYER = np.dtype([("weight", "<u8"), ("bias", "<u8"), ("rows", "<i4"), ("offset", "<i4"), ("row", "<i4"),
                         ("scale", "<f4"), ("bias_scale", "<f4"), ("pad", "<i4")])   # svbrdf_style_layer


class StyleLayersFunction(torch.autograd.Function):
    """Every style layer of a synthesis pass in one launch: latent [1, L, dim],
    the layers' weights [rows, dim] and biases [rows] and (latent row, scale,
    bias scale) of each -> the styles side by side, [sum of rows].  The
    weights are frozen; the backward gives dL/dlatent."""

    @staticmethod
    def _table(weights, biases, layers):
        rows = [int(w.shape[0]) for w in weights]
        table = np.zeros(len(weights), _STYLE_LAYER)
        table["weight"] = [w.data_ptr() for w in weights]
        table["bias"] = [b.data_ptr() for b in biases]
        table["rows"] = rows
        table["offset"] = np.cumsum([0] + rows[:-1])
        table["row"], table["scale"], table["bias_scale"] = zip(*layers)
        return table

    @staticmethod
    def forward(ctx, latent, weights, biases, layers):
        x = latent.detach().contiguous()
        if x.data_ptr() % 16:   # a view at an odd offset: the kernel reads 16 bytes at a time
            x = x.clone()
        table = StyleLayersFunction._table(weights, biases, layers)
        out = torch.empty(int(table["rows"].sum()), dtype=torch.float32, device=x.device)
        _lib.call("svbrdf_style_layers", table.ctypes.data, len(weights), _lib.ptr(x), int(x.shape[1]),
                  int(x.shape[2]), _lib.ptr(out), _lib.stream_handle(x.device))
        ctx.save_for_backward(*weights)
        ctx.layers, ctx.shape = layers, tuple(x.shape)
        return out

    @staticmethod
    def backward(ctx, grad):
        g = grad.contiguous()
        weights = ctx.saved_tensors
        table = StyleLayersFunction._table(weights, weights, ctx.layers)   # the biases are not read
        _, n_rows, dim = ctx.shape
        nb = int(_lib.query("svbrdf_style_layers_grad_workspace_bytes", table.ctypes.data, len(weights), dim))
        ws = torch.empty(nb // 4, dtype=torch.float32, device=g.device)
        out = torch.empty(ctx.shape, dtype=torch.float32, device=g.device)
        _lib.call("svbrdf_style_layers_grad", table.ctypes.data, len(weights), _lib.ptr(g), n_rows, dim, _lib.ptr(out),
                  _lib.ptr(ws), nb, _lib.stream_handle(g.device))
        return out, None, None, None


class ToRGBFunction(torch.autograd.Function):
    """The 1x1 output convolution of one sample, its weight [cout, cin, 1, 1]
    (frozen) scaled per input channel by style * scale, plus the upsampled
    skip image (or None)."""

    @staticmethod
    def forward(ctx, x, style, weight, scale, skip):
        x = x.contiguous()
        st, wt = style.detach().contiguous(), weight.detach().contiguous()
        sk = None if skip is None else skip.detach().contiguous()
        for t, name in ((x, "x"), (st, "style"), (wt, "weight"), *(() if sk is None else ((sk, "skip"),))):
            _check(t, name)
        n, cin, h, w = (int(s) for s in x.shape)
        cout = int(wt.shape[0])
        if n != 1 or tuple(wt.shape) != (cout, cin, 1, 1) or st.numel() != cin:
            raise ValueError(f"x {tuple(x.shape)}, weight {tuple(wt.shape)} and style {st.numel()} do not match")
        if sk is not None and tuple(sk.shape) != (1, cout, h // 2, w // 2):
            raise ValueError(f"skip {tuple(sk.shape)} is not half of [1, {cout}, {h}, {w}]")
        y = torch.empty((1, cout, h, w), dtype=torch.float32, device=x.device)
        _lib.call("svbrdf_torgb", _lib.ptr(x), cin, h, w, _lib.ptr(wt), cout, _lib.ptr(st), float(scale), _lib.ptr(sk),
                  _lib.ptr(y), _lib.stream_handle(x.device))
        ctx.save_for_backward(x, style, weight)
        ctx.scale = float(scale)
        return y

    @staticmethod
    def backward(ctx, grad_y):
        x, style, weight = ctx.saved_tensors
        g = grad_y.contiguous()
        cout, cin = int(weight.shape[0]), int(weight.shape[1])
        gm, wm = g.view(cout, -1), weight.view(cout, cin)
        gx = gs = gskip = None
        if ctx.needs_input_grad[0]:
            gx = torch.mm((wm * (style.reshape(1, cin) * ctx.scale)).t(), gm).view(x.shape)
        if ctx.needs_input_grad[1]:
            gs = ((torch.mm(gm, x.view(cin, -1).t()) * wm).sum(dim=0) * ctx.scale).reshape(style.shape)
        if ctx.needs_input_grad[4]:
            gskip = Upsample2Function.adjoint(g)
        return gx, gs, None, None, gskip


class Upsample2Function(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x):
        x = x.contiguous()
        _check(x, "x")
        n, c, h, w = (int(s) for s in x.shape)
        y = torch.empty((n, c, 2 * h, 2 * w), dtype=torch.float32, device=x.device)
        _lib.call("svbrdf_upsample2_blur", _lib.ptr(x), n * c, h, w, _lib.ptr(y), _lib.stream_handle(x.device))
        return y

    @staticmethod
    def backward(ctx, grad_y):
        return Upsample2Function.adjoint(grad_y)

    @staticmethod
    def adjoint(grad_y):
        g = grad_y.contiguous()
        n, c, h2, w2 = (int(s) for s in g.shape)
        gx = torch.empty((n, c, h2 // 2, w2 // 2), dtype=torch.float32, device=g.device)
        _lib.call("svbrdf_upsample2_blur_adjoint", _lib.ptr(g), n * c, h2 // 2, w2 // 2, _lib.ptr(gx),
                  _lib.stream_handle(g.device))
        return gx


def upsample2(x):
    return Upsample2Function.apply(x)


class AvgPool2Function(torch.autograd.Function):
    """F.avg_pool2d(x, 2) (src/descriptor.py:15-18 puts AvgPool2d(2) in
    place of VGG's max pooling) on the HIP kernels: same bits forward, and
    the adjoint writes dL/dy / 4 to each window."""

    @staticmethod
    def forward(ctx, x):
        x = x.contiguous()
        _check(x, "x")
        n, c, h, w = (int(s) for s in x.shape)
        y = torch.empty((n, c, h // 2, w // 2), dtype=torch.float32, device=x.device)
        _lib.call("svbrdf_avgpool2", _lib.ptr(x), n * c, h, w, _lib.ptr(y), _lib.stream_handle(x.device))
        ctx.shape = (n, c, h, w)
        return y

    @staticmethod
    def backward(ctx, grad_y):
        g = grad_y.contiguous()
        n, c, h, w = ctx.shape
        gx = torch.empty((n, c, h, w), dtype=torch.float32, device=g.device)
        _lib.call("svbrdf_avgpool2_adjoint", _lib.ptr(g), n * c, h, w, _lib.ptr(gx), _lib.stream_handle(g.device))
        return gx


def avgpool2(x):
    return AvgPool2Function.apply(x)


class _FrozenConvFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, layer, tap=None, tap_scale=1.0):
        n, _, h, w = x.shape
        split = layer.split if _takes_split(n, layer.cin, h, w, layer.cout) else None   # None below 32 channels
        y = _conv3x3(x, layer.packed, split, layer.cin, layer.cout, layer.bias, None, 0.0, layer.act, tap, tap_scale)
        ctx.save_for_backward(y)
        ctx.layer = layer
        return y

    @staticmethod
    def backward(ctx, grad_y):
        (y,) = ctx.saved_tensors
        layer = ctx.layer
        n, cout, h, w = y.shape
        split_t = layer.split_t if _takes_split(n, cout, h, w, layer.cin) else None
        return _input_grad(grad_y, y, layer.packed_t, split_t, layer.cin, layer.act), None, None, None


class _PooledConvFunction(torch.autograd.Function):
    """Conv3x3 and the 2x2 average pooling behind it, outside autograd: the
    pooled output, and the output itself where `keep`."""

    @staticmethod
    def forward(ctx, x, layer, keep, tap, tap_scale):
        n, channels, h, w = (int(s) for s in x.shape)
        x, bias, _ = _conv_inputs(x, layer.bias, None)
        shape = (n, layer.cout, h, w)
        y = torch.empty(shape, dtype=torch.float32, device=x.device) if keep else None
        if tap is not None:
            _check_tap(tap, x, n * layer.cout * h * w)
        pool = torch.empty((n, layer.cout, h // 2, w // 2), dtype=torch.float32, device=x.device)
        _lib.call("svbrdf_conv3x3_pooled", _lib.ptr(x), n, channels, h, w, _lib.ptr(layer.split), layer.cout,
                  _lib.ptr(bias), None, 0.0, ACT[layer.act], _lib.ptr(y), _lib.ptr(tap), float(tap_scale),
                  _lib.ptr(pool), _lib.stream_handle(x.device))
        return (pool, y) if keep else pool


class Conv3x3(torch.nn.Module):
    """A 3x3 layer with frozen weights [Cout, Cin, 3, 3] and bias [Cout],
    followed by `act`: packed once in the forward and input-gradient layouts."""

    def __init__(self, weight, bias=None, act="relu"):
        super().__init__()
        if act not in ACT:
            raise ValueError(f"act must be one of {sorted(ACT)}")
        self.cout, self.cin = int(weight.shape[0]), int(weight.shape[1])
        self.weight = weight.detach().contiguous()
        self.bias = None if bias is None else bias.detach().contiguous()
        self.act = act
        self.packed = pack3x3(self.weight)
        self.packed_t = pack3x3(self.weight, transpose=True)
        self._splits = {name: (t, _version(t), _split_packed(t))
                        for name, t in (("packed", self.packed), ("packed_t", self.packed_t))
                        if min(self.cin, self.cout) >= 32}

    _splits = {}   # of a layer that was saved without any

    def _split(self, name):
        """The layout of the bf16 matrix cores of self.packed or self.packed_t,
        for the sizes that take that path; None below 32 channels on either
        side.  Kept with the tensor it was made from, and made again once that
        one has been replaced or written to."""
        if min(self.cin, self.cout) < 32:
            return None
        packed = getattr(self, name)
        source, seen, split = self._splits.get(name, (None, None, None))
        if source is packed and seen == _version(packed):
            return split
        _check(packed, name)
        shape = (9, self.cin, self.cout) if name == "packed" else (9, self.cout, self.cin)
        if tuple(packed.shape) != shape:
            raise ValueError(f"{name} {tuple(packed.shape)} is not {shape}")
        split = _split_packed(packed)
        if not torch.cuda.is_current_stream_capturing():
            # whole before another stream can find it
            torch.cuda.current_stream(packed.device).synchronize()
            self._splits = {**self._splits, name: (packed, _version(packed), split)}
        return split

    @property
    def split(self):
        return self._split("packed")

    @property
    def split_t(self):
        return self._split("packed_t")

    def forward(self, x, tap=None, tap_scale=1.0):
        """The layer; tap: a flat tensor that also receives tap_scale times
        the output, outside autograd only."""
        if tap is None:
            return _FrozenConvFunction.apply(x, self)
        if torch.is_grad_enabled() and x.requires_grad:
            raise ValueError("tap is written outside autograd: not with an input that requires a gradient")
        return _FrozenConvFunction.apply(x, self, tap, tap_scale)

    def pooled(self, x, keep=True, tap=None, tap_scale=1.0):
        """(avgpool2(output), output): outside autograd in one kernel where the
        shape allows it (svbrdf_conv3x3_split_pools), the output then written
        only where `keep` (else None); tap as in forward."""
        n, channels, h, w = x.shape
        if (self.split is None or channels != self.cin or (torch.is_grad_enabled() and x.requires_grad)
                or not _lib.query("svbrdf_conv3x3_split_pools", n, channels, h, w, self.cout)):
            y = self(x, tap, tap_scale)
            return avgpool2(y), y
        if keep:
            return _PooledConvFunction.apply(x, self, True, tap, tap_scale)
        return _PooledConvFunction.apply(x, self, False, tap, tap_scale), None
