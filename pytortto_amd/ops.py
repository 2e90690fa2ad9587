"""Typed Python wrappers over the C ABI, operating on ``hiparray`` device arrays.

Shape bookkeeping and output allocation happen here; all arithmetic happens in
``libtortto_hip.so``.  Each wrapper names the reference lines whose array expressions it
stands in for (paths relative to the reference's ``src/tortto/``).
"""
import ctypes
import functools
import math
import weakref
from math import prod

import numpy as np

from . import _hip
from .xparray import hiparray, poison


_F32 = np.dtype(np.float32)


def _ptr(a):
    return None if a is None else a.ptr


def _f32(*arrays):
    for a in arrays:
        if a is not None and a.dtype is not _F32 and a.dtype != _F32:
            raise TypeError(f'the device path computes in float32 only, got {a.dtype}')


def computes_on(*arrays):
    """Whether the device path takes all of them (None: not given) as operands."""
    for a in arrays:
        if a is not None and (a.__class__ is not hiparray or a._dtype is not _F32 and a._dtype != _F32):
            return False
    return True


def conv_out_size(size, k, stride, pad, dil):
    """autograd/grad_nn.py:565-566"""
    return math.floor((size + 2 * pad - dil * (k - 1) - 1) / stride + 1)


@functools.lru_cache(maxsize=1024, typed=True)
def _conv2d_shapes(n, c, h, wd, k, cg, r, s, sh, sw, ph, pw, dh, dw, groups):
    """(shape of y, the C entry points' integer arguments); p or q may be empty."""
    p, q = conv_out_size(h, r, sh, ph, dh), conv_out_size(wd, s, sw, pw, dw)
    return (n, k, p, q), (n, c, h, wd, k, r, s, sh, sw, ph, pw, dh, dw, groups)


# ---- convolution -------------------------------------------------------------------------------

def _conv2d_geometry(x, w, bias, stride, padding, dilation, groups):
    """(shape of y, the C entry points' integer arguments); raises for an empty output."""
    _f32(x, w, bias)
    n, c, h, wd = x.shape
    k, cg, r, s = w.shape
    shape, dims = _conv2d_shapes(n, c, h, wd, k, cg, r, s, stride[0], stride[1], padding[0], padding[1], dilation[0],
                                 dilation[1], groups)
    p, q = shape[2:]
    if p <= 0 or q <= 0:
        raise RuntimeError(f'Calculated output size ({k} x {p} x {q}) is too small for input {x.shape} '
                           f'and kernel {(r, s)}')
    return shape, dims


def conv2d_fwd(x, w, bias, stride, padding, dilation, groups):
    """y = conv(x, w) + bias  (autograd/grad_nn.py:595-643, :709-711)."""
    shape, dims = _conv2d_geometry(x, w, bias, stride, padding, dilation, groups)
    y = hiparray.empty(shape)
    _hip.call('tt_conv2d_fwd_f32', x.ptr, w.ptr, _ptr(bias), y.ptr, *dims)
    return y


_BN_CHANNELS = 65535        # of the BatchNorm entry points


class DeferredConv:
    """A convolution whose result needs no gradient, not launched yet (see ``_hip.defer``).  What
    follows it in an evaluation pass -- a BatchNorm with given statistics, a residual add, a ReLU --
    joins the launch and is applied to the accumulators before they are stored (``absorb_norm``,
    ``absorb_add``, ``run_with_relu``, in this order); anything else finds it launched with what has joined so far.

    A value in between that nobody holds any more when the launch comes is never stored.  One that is still
    held may be read (a shortcut around the BatchNorm): it is stored where it stands, and what follows it runs
    in kernels of its own (same bits), so that no convolution is ever computed twice.  The ReLU is parked with the
    rest, and all of it stays parked behind the next convolution until a third, or another call, comes: by then the
    caller's names for the values in front are mostly gone."""
    queues = True

    def __init__(self, x, w, bias, shape, dims):
        self.x, self.w, self.bias, self.dims = x, w, bias, dims
        self.norm = self.residual = None
        self.steps = []         # what has joined
        self.shape = shape
        self.out = hiparray.lazy(self.shape)
        self.between = []       # (a weak reference to the buffer of a value in front of ``out``, steps in front of it)

    def _join(self, step, out):
        if out is not None:
            self.between.append((weakref.ref(self.out._buf), len(self.steps)))
            self.out = out
        self.steps.append(step)
        _hip.defer(self)
        return self.out

    def takes_norm(self):
        return not self.steps and self.shape[1] <= _BN_CHANNELS

    def takes_add(self):
        return self.residual is None and self.takes_relu()

    def takes_relu(self):
        return 'relu' not in self.steps

    def absorb_norm(self, mean, var, gamma, beta, eps):
        self.norm = (mean, var, gamma, beta, float(eps))
        return self._join('norm', hiparray.lazy(self.shape))

    def absorb_add(self, residual):
        self.residual = residual
        return self._join('add', hiparray.lazy(self.shape))

    def run_with_relu(self, out=None):
        """The ReLU's values go to ``out``, or to the operation's own array (an in-place ReLU)."""
        return self._join('relu', out)

    def _held(self):
        """(array, steps in front of it) of the values in between that somebody still holds."""
        buffers = [(ref(), done) for ref, done in self.between]
        return [(hiparray.on(buf, self.shape, self.out.dtype), done) for buf, done in buffers if buf is not None]

    def run(self):
        before = None
        for array, done in (*self._held(), (self.out, len(self.steps))):
            if before is None:
                self._launch(array, self.steps[:done])
            else:
                self._launch_after(before[0], array, self.steps[before[1]:done])
            before = array, done

    def _launch(self, out, steps):
        """The convolution and the ``steps`` behind it, in one launch."""
        x, w, bias, dims = self.x, self.w, self.bias, self.dims
        if not steps:
            _hip.call('tt_conv2d_fwd_f32', x.ptr, w.ptr, _ptr(bias), out.ptr, *dims)
            return
        mean, var, gamma, beta, eps = self.norm if 'norm' in steps else (None, None, None, None, 0.0)
        residual = self.residual if 'add' in steps else None
        _hip.call('tt_conv2d_norm_act_fwd_f32', x.ptr, w.ptr, _ptr(bias), out.ptr, _ptr(mean), _ptr(var), _ptr(gamma),
                  _ptr(beta), eps, _ptr(residual), int('relu' in steps), *dims)

    def _launch_after(self, value, out, steps):
        """``steps`` on a value that has been stored."""
        relu = 'relu' in steps
        if 'norm' in steps:
            mean, var, gamma, beta, eps = self.norm
            add = 'add' in steps
            op = DeferredBatchNormEval(value, gamma, beta, mean, var, eps, None if add else out)
            op.launch(relu and not add)
            if not add:
                return
            value = op.out
        if 'add' in steps:
            _hip.call('tt_add_relu_f32' if relu else 'tt_add_f32', value.ptr, self.residual.ptr, out.ptr, out.size)
        else:
            _hip.call('tt_relu_fwd_f32', value.ptr, out.ptr, out.size)

    def poison(self, exc):
        poison([self.out] + [array for array, _ in self._held()], exc)


@functools.lru_cache(maxsize=1024, typed=True)
def _conv2d_fwd_accepts(elements, *dims):
    """Whether the C entry point takes this geometry, by its own argument checks (the size query runs them and
    launches nothing), in one run of images (the larger tensor's ``elements`` say so); asked once per geometry."""
    if 0 in dims[:4] or elements >= 1 << 31:
        return False
    try:
        return _hip.lib().tt_workspace_size_conv2d_fwd_f32(ctypes.byref(ctypes.c_size_t()), *dims) == 0
    except ctypes.ArgumentError:
        return False


def conv2d_fwd_deferred(x, w, bias, stride, padding, dilation, groups):
    """``conv2d_fwd`` with the launch parked for the operations behind it to join.  What would be refused is
    launched at once, so that the error is raised where it belongs, and so is a batch that is cut into runs."""
    shape, dims = _conv2d_geometry(x, w, bias, stride, padding, dilation, groups)
    if not _conv2d_fwd_accepts(max(prod(x.shape), prod(shape)), *dims):
        return conv2d_fwd(x, w, bias, stride, padding, dilation, groups)
    op = DeferredConv(x, w, bias, shape, dims)
    _hip.defer(op)
    return op.out


def conv2d_dgrad(dy, w, bias, out_hw, stride, padding, dilation, groups, add=None, relu_y=None):
    """dx = sum_k,r,s dy * w  for a conv weight ``w[K, C/g, R, S]`` (autograd/grad_nn.py:659-682).
    ``out_hw`` is the spatial size of the result; ``bias`` (length C) is added when given
    (transposed-convolution forward, grad_nn.py:755-757).  At stride 1 without a bias, ``add`` (what
    has already arrived for x) is added to dx, and the sum multiplied by ``relu_y > 0``."""
    _f32(dy, w, bias, add, relu_y)
    n, k, p, q = dy.shape
    _, cg, r, s = w.shape
    c = cg * groups
    hx, wx = out_hw
    dx = hiparray.empty((n, c, hx, wx))
    dims = (n, c, hx, wx, k, r, s, stride[0], stride[1], padding[0], padding[1], dilation[0], dilation[1], groups, p, q)
    if add is None and relu_y is None:
        _hip.call('tt_conv2d_dgrad_f32', dy.ptr, w.ptr, _ptr(bias), dx.ptr, *dims)
    else:
        _hip.call('tt_conv2d_dgrad_acc_f32', dy.ptr, w.ptr, dx.ptr, _ptr(add), _ptr(relu_y), *dims)
    return dx


def conv2d_wgrad(x, dy, w_shape, stride, padding, dilation, groups):
    """dw = sum_n,p,q x~ * dy  (autograd/grad_nn.py:646-656)."""
    _f32(x, dy)
    n, c, h, wd = x.shape
    _, k, p, q = dy.shape
    r, s = w_shape[-2:]
    dw = hiparray.empty(tuple(w_shape))
    _hip.call('tt_conv2d_wgrad_f32', x.ptr, dy.ptr, dw.ptr, n, c, h, wd, k, r, s,
              stride[0], stride[1], padding[0], padding[1], dilation[0], dilation[1], groups, p, q)
    return dw


def channel_sum(t):
    """t.sum((0, 2, 3)) for an NCHW array (autograd/grad_nn.py:728, :774)."""
    _f32(t)
    n, k = t.shape[:2]
    hw = t.size // (n * k) if n * k else 0
    out = hiparray.empty((k,))
    _hip.call('tt_channel_sum_f32', t.ptr, out.ptr, n, k, hw)
    return out


# ---- BatchNorm ---------------------------------------------------------------------------------

def _nchw(x):
    n, c = x.shape[:2]
    return n, c, x.size // (n * c) if n * c else 0


def bn_fwd_train(x, gamma, beta, running_mean, running_var, momentum, eps, num_batches_tracked=None):
    """Training forward (autograd/grad_nn.py:921-930, :942-959).  Returns
    ``(y, mean, var_eps, sd, new_running_mean, new_running_var)``; the last two are new arrays
    (``None`` without running statistics), as the reference rebinds ``.data``.
    ``num_batches_tracked`` (a one-element device array) is incremented by one in the same launch:
    the module's ``num_batches_tracked.data += 1`` (nn/modules/batchnorm.py:66)."""
    _f32(x, gamma, beta, running_mean, running_var)
    n, c, hw = _nchw(x)
    y = hiparray.empty(x.shape)
    mean, var_eps, sd = hiparray.empty((c,)), hiparray.empty((c,)), hiparray.empty((c,))
    track = running_mean is not None and running_var is not None
    new_rm = hiparray.empty((c,)) if track else None
    new_rv = hiparray.empty((c,)) if track else None
    _hip.call('tt_bn_fwd_train_f32', x.ptr, _ptr(gamma), _ptr(beta), y.ptr, mean.ptr, var_eps.ptr, sd.ptr,
              _ptr(running_mean) if track else None, _ptr(running_var) if track else None,
              _ptr(new_rm), _ptr(new_rv), _ptr(num_batches_tracked),
              float(momentum if momentum is not None else 0.0), float(eps), n, c, hw)
    return y, mean, var_eps, sd, new_rm, new_rv


class DeferredBatchNorm:
    """A training forward that has not been launched yet (see ``_hip.defer``).  What follows may join
    the launch: a residual added to the normalised values (``absorb_add``) and a ReLU
    (``run_with_relu(out)``: the output is ``maximum(., 0)``, in ``out``, or in the operation's own array
    when ``out`` is None, an in-place ReLU); ``run()`` launches what has joined so far.
    The values in between are then never stored: their arrays recompute them (same kernels, same bits,
    scratch statistics, no running update) should anybody ask, and at the latest just before an operand
    is written in place: what is read back is always what the reference stored when the operation ran."""

    def __init__(self, x, gamma, beta, running_mean, running_var, momentum, eps, num_batches_tracked):
        self.x, self.gamma, self.beta = x, gamma, beta
        self.momentum, self.eps = float(momentum if momentum is not None else 0.0), float(eps)
        self.nbt = num_batches_tracked
        self.dims = n, c, hw = _nchw(x)
        self.residual = None
        self.out = self.y = hiparray.lazy(x.shape)
        self.stats = [hiparray.empty((c,)) for _ in range(3)]        # mean, var + eps, sd
        self.track = running_mean is not None and running_var is not None
        self.rm_in, self.rv_in = (running_mean, running_var) if self.track else (None, None)
        self.new_rm = hiparray.empty((c,)) if self.track else None
        self.new_rv = hiparray.empty((c,)) if self.track else None

    def _launch(self, out, relu, coef=None):
        mean, var_eps, sd = self.stats
        _hip.call('tt_bn_act_fwd_train_f32', self.x.ptr, _ptr(self.gamma), _ptr(self.beta), _ptr(self.residual), out.ptr,
                  mean.ptr, var_eps.ptr, sd.ptr, _ptr(coef), _ptr(self.rm_in), _ptr(self.rv_in), _ptr(self.new_rm),
                  _ptr(self.new_rv), _ptr(self.nbt), self.momentum, self.eps, int(relu), *self.dims)

    def _on_demand(self):
        """The output so far is about to be absorbed: leave it to be recomputed on demand."""
        x, gamma, beta, residual, eps, dims = self.x, self.gamma, self.beta, self.residual, self.eps, self.dims

        def recompute(buf):
            scratch = [hiparray.empty((dims[1],)) for _ in range(3)]
            _hip.call('tt_bn_act_fwd_train_f32', x.ptr, _ptr(gamma), _ptr(beta), _ptr(residual), buf.ptr, scratch[0].ptr,
                      scratch[1].ptr, scratch[2].ptr, None, None, None, None, None, None, 0.0, eps, 0, *dims)
        # the operands as they are now: should one of them be written in place later (an optimiser step,
        # ``+=``), the values are produced first
        self.out._buf.fill_on_demand(recompute, (x, gamma, beta, residual))

    def run(self):
        self._launch(self.out, False)

    def takes_add(self):
        return self.residual is None

    def absorb_add(self, residual):
        self._on_demand()
        self.residual = residual
        self.out = hiparray.lazy(self.out.shape)
        _hip.defer(self)
        return self.out

    def run_with_relu(self, out=None, keep_coef=False):
        """With ``keep_coef`` the channels' two constants stay in ``coef``, for the backward to apply the
        ReLU's mask from x alone (only without a residual in between)."""
        self.coef = hiparray.empty((2 * self.dims[1],)) if keep_coef and self.residual is None else None
        if out is None:
            out = self.out
            self._launch(out, True, self.coef)
        else:
            self._launch(out, True, self.coef)
            self._on_demand()
        return out

    def poison(self, exc):
        poison([self.y, self.out, *self.stats, self.new_rm, self.new_rv], exc)


def bn_fwd_train_deferred(x, gamma, beta, running_mean, running_var, momentum, eps, num_batches_tracked=None):
    """``bn_fwd_train`` with the launch parked for the next operation to absorb (a ReLU) or to
    trigger (anything else).  Same return value; the arrays are filled when the launch happens."""
    _f32(x, gamma, beta, running_mean, running_var)
    op = DeferredBatchNorm(x, gamma, beta, running_mean, running_var, momentum, eps, num_batches_tracked)
    _hip.defer(op)
    return (op.y, *op.stats, op.new_rm, op.new_rv)


class DeferredReluBackward:
    """``dy * (y > 0)`` not launched yet: the backward of the BatchNorm the ReLU was fused with forms the
    product itself while it reads ``dy`` (``bn_bwd`` with ``coef``, the constants that forward kept);
    anything else finds it computed."""

    def __init__(self, dy, y, coef):
        self.dy, self.y, self.coef = dy, y, coef
        self.out = hiparray.lazy(y.shape)

    def run(self):
        _hip.call('tt_relu_bwd_f32', self.dy.ptr, self.y.ptr, self.out.ptr, self.y.size)

    def poison(self, exc):
        poison([self.out], exc)


def relu_bwd_deferred(dy, y, coef):
    _f32(dy, y)
    op = DeferredReluBackward(dy, y, coef)
    _hip.defer(op)
    return op.out


class DeferredBatchNormEval:
    """Normalisation with given statistics (autograd/grad_nn.py:931-959), not launched yet: a ReLU that
    comes next is applied in the same pass, as ``DeferredBatchNorm`` has it for training."""

    def __init__(self, x, gamma, beta, mean_in, var_in, eps, out=None, keep_stats=False):
        self.operands = (x, gamma, beta, mean_in, var_in)
        self.eps, self.dims = float(eps), _nchw(x)
        self.out = hiparray.lazy(x.shape) if out is None else out
        self.stats = [hiparray.empty((self.dims[1],)) for _ in range(3)] if keep_stats else []   # mean, var + eps, sd

    def _launch(self, entry, out):
        x, gamma, beta, mean_in, var_in = self.operands
        if self.stats:
            stats = [a.ptr for a in self.stats]
        else:                                               # nobody reads them
            scratch, step = hiparray.empty((3 * self.dims[1],)), 4 * self.dims[1]
            stats = [scratch.ptr, scratch.ptr + step, scratch.ptr + 2 * step]
        _hip.call(entry, x.ptr, _ptr(gamma), _ptr(beta), out.ptr, mean_in.ptr, var_in.ptr, *stats, self.eps, *self.dims)

    def launch(self, relu):
        self._launch('tt_bn_relu_fwd_eval_f32' if relu else 'tt_bn_fwd_eval_f32', self.out)

    def run(self):
        self.launch(False)

    def run_with_relu(self, out=None):
        if out is None:
            out = self.out
        else:
            self.out._buf.fill_on_demand(lambda buf: self._launch('tt_bn_fwd_eval_f32', buf), self.operands)
        self._launch('tt_bn_relu_fwd_eval_f32', out)
        return out

    def poison(self, exc):
        poison([self.out, *self.stats], exc)


def bn_fwd_eval(x, gamma, beta, mean_in, var_in, eps, deferred=False):
    """[y, mean, var + eps, sd]; with ``deferred`` [y], whose launch is parked for a ReLU to join, unless it would
    be refused: that error is raised here."""
    _f32(x, gamma, beta, mean_in, var_in)
    op = DeferredBatchNormEval(x, gamma, beta, mean_in, var_in, eps, keep_stats=not deferred)
    n, c, hw = op.dims
    if deferred and n and hw and 0 < c <= _BN_CHANNELS and max(n, c) * hw < 1 << 31 and computes_on(*op.operands):
        _hip.defer(op)
    else:
        op.run()
    return [op.out, *op.stats]


def bn_bwd(x, dy, gamma, mean, var_eps, sd, need=(True, True, True), coef=None, add=None):
    """Backward (autograd/grad_nn.py:966-989): returns ``(dx, dgamma, dbeta)``.  With ``coef`` the gradient
    is ``dy * (bn(x) > 0)``, masked as it is read (a fused ReLU's backward); ``add`` (what has already
    arrived for x) is added to dx."""
    _f32(x, dy, gamma, add)
    n, c, hw = _nchw(x)
    dx = hiparray.empty(x.shape) if need[0] else None
    dgamma = hiparray.empty((c,)) if need[1] else None
    dbeta = hiparray.empty((c,)) if need[2] else None
    _hip.call('tt_bn_act_bwd_f32', x.ptr, dy.ptr, _ptr(coef), _ptr(gamma), mean.ptr, var_eps.ptr, sd.ptr,
              _ptr(dx), _ptr(add), _ptr(dgamma), _ptr(dbeta), n, c, hw)
    return dx, dgamma, dbeta


# ---- elementwise glue ----------------------------------------------------------------------------

def relu_fwd(x, out=None):
    _f32(x)
    y = hiparray.empty(x.shape) if out is None else out.own()
    _hip.call('tt_relu_fwd_f32', x.ptr, y.ptr, x.size)
    return y


def relu_bwd(dy, y):
    _f32(dy, y)
    dx = hiparray.empty(y.shape)
    _hip.call('tt_relu_bwd_f32', dy.ptr, y.ptr, dx.ptr, y.size)
    return dx


def leaky_relu_fwd(x, negative_slope, out=None):
    _f32(x)
    y = hiparray.empty(x.shape) if out is None else out.own()
    _hip.call('tt_leaky_relu_fwd_f32', x.ptr, y.ptr, float(negative_slope), x.size)
    return y


def leaky_relu_bwd(dy, x, negative_slope, out=None):
    _f32(dy, x)
    dx = hiparray.empty(x.shape) if out is None else out.own()
    _hip.call('tt_leaky_relu_bwd_f32', dy.ptr, x.ptr, dx.ptr, float(negative_slope), x.size)
    return dx


def add(a, b):
    _f32(a, b)
    if a.shape != b.shape:
        raise ValueError(f'device add needs equal shapes, got {a.shape} and {b.shape}')
    out = hiparray.empty(a.shape)
    _hip.call('tt_add_f32', a.ptr, b.ptr, out.ptr, a.size)
    return out


class DeferredAdd:
    """``a + b`` of equal shapes, not launched yet (see ``_hip.defer``): a ReLU that comes next
    computes ``maximum(a + b, 0)`` in one pass (``run_with_relu``); anything else finds the sum done.
    When the ReLU's result went to an array of its own, the sum itself is produced on demand -- at the
    latest just before ``a`` or ``b`` is written in place."""

    def __init__(self, a, b):
        self.a, self.b = a, b
        self.out = hiparray.lazy(a.shape)

    def run(self):
        _hip.call('tt_add_f32', self.a.ptr, self.b.ptr, self.out.ptr, self.a.size)

    def run_with_relu(self, out=None):
        a, b = self.a, self.b
        if out is None:
            _hip.call('tt_add_relu_f32', a.ptr, b.ptr, self.out.ptr, a.size)
            return self.out
        _hip.call('tt_add_relu_f32', a.ptr, b.ptr, out.ptr, a.size)
        self.out._buf.fill_on_demand(lambda buf: _hip.call('tt_add_f32', a.ptr, b.ptr, buf.ptr, a.size), (a, b))
        return out

    def poison(self, exc):
        poison([self.out], exc)


def add_deferred(a, b):
    _f32(a, b)
    if a.shape != b.shape:
        raise ValueError(f'device add needs equal shapes, got {a.shape} and {b.shape}')
    op = DeferredAdd(a, b)
    _hip.defer(op)
    return op.out


# ---- MaxPool2d -------------------------------------------------------------------------------------

def _pool_dims(x):
    if x.ndim not in (3, 4):
        raise ValueError(f'max pooling needs [N,C,H,W] or [C,H,W] planes, got shape {x.shape}')
    return prod(x.shape[:-2]), x.shape[-2], x.shape[-1]


def maxpool2d_fwd(x, out_hw, kernel_size, stride, padding, dilation):
    """(y, tap): maxima over the -inf padded windows and, per output, the winning tap as
    kernel_row * kw + kernel_column (``_max_pool2d``, grad_nn.py:784-808): a byte each where that fits."""
    _f32(x)
    nc, h, w = _pool_dims(x)
    p, q = out_hw
    y = hiparray.empty(x.shape[:-2] + (p, q))
    byte = kernel_size[0] * kernel_size[1] <= 256
    tap = hiparray.empty(x.shape[:-2] + (p, q), np.uint8 if byte else np.int32)
    _hip.call('tt_maxpool2d_fwd_tap8_f32' if byte else 'tt_maxpool2d_fwd_f32', x.ptr, y.ptr, tap.ptr, nc, h, w, p, q, *kernel_size, *stride, *padding,
              *dilation)
    return y, tap


def maxpool2d_bwd(dy, tap, in_hw, kernel_size, stride, padding, dilation):
    """dx: every output gradient assigned to its window's arg-max pixel, the last window in
    (p, q) order winning where several chose the same pixel (``_max_pool2d_backward``, :811-824)."""
    _f32(dy)
    if tap.dtype not in (np.uint8, np.int32) or tap.shape != dy.shape:
        raise ValueError('maxpool2d_bwd: `tap` must be the array the forward returned')
    nc, p, q = _pool_dims(dy)
    h, w = in_hw
    dx = hiparray.empty(dy.shape[:-2] + (h, w))
    _hip.call('tt_maxpool2d_bwd_tap8_f32' if tap.dtype == np.uint8 else 'tt_maxpool2d_bwd_f32', dy.ptr, tap.ptr, dx.ptr, nc, h, w, p, q, *kernel_size, *stride, *padding,
              *dilation)
    return dx


# ---- classifier head -----------------------------------------------------------------------------

def mean_trailing(x, k, keepdim):
    """Mean over the last ``k`` dimensions (autograd/grad_fcn.py:1058-1067)."""
    _f32(x)
    lead, tail = x.shape[:-k], x.shape[-k:]
    y = hiparray.empty(lead + ((1,) * k if keepdim else ()))
    _hip.call('tt_mean_rows_f32', x.ptr, y.ptr, prod(lead), prod(tail))
    return y


def mean_trailing_bwd(g, x_shape, k):
    """The gradient divided by the element count and repeated over the reduced dimensions
    (grad_fcn.py:1069-1093); materialised, where the reference returns a stride-0 view."""
    _f32(g)
    dx = hiparray.empty(x_shape)
    _hip.call('tt_mean_rows_bwd_f32', g.ptr, dx.ptr, prod(x_shape[:-k]), prod(x_shape[-k:]))
    return dx


def transpose2d(x):
    _f32(x)
    r, c = x.shape
    y = hiparray.empty((c, r))
    _hip.call('tt_transpose2d_f32', x.ptr, y.ptr, r, c)
    return y


_ONE = ((1, 1), (0, 0), (1, 1), 1)   # stride, padding, dilation, groups of a plain matrix product


def mm(a, b):
    """a[M,K] @ b[K,N] (grad_fcn.py:907-918) on the implicit-GEMM convolution kernel: b is the
    image [1, K, 1, N], a the 1x1 weights [M, K, 1, 1]."""
    (m, k), (k2, n) = a.shape, b.shape
    if k != k2:
        raise RuntimeError(f'mat1 and mat2 shapes cannot be multiplied ({m}x{k} and {k2}x{n})')
    return conv2d_fwd(b.reshape((1, k, 1, n)), a.reshape((m, k, 1, 1)), None, *_ONE).reshape((m, n))


def mm_grad_a(g, b):
    """g[M,N] @ b[K,N].T (grad_fcn.py:927-928): the weight gradient of the same 1x1 geometry."""
    (m, n), (k, _) = g.shape, b.shape
    return conv2d_wgrad(b.reshape((1, k, 1, n)), g.reshape((1, m, 1, n)), (m, k, 1, 1), *_ONE).reshape((m, k))


def mm_grad_b(a, g):
    """a[M,K].T @ g[M,N] (grad_fcn.py:929-930): the input gradient of the same 1x1 geometry."""
    (m, k), (_, n) = a.shape, g.shape
    return conv2d_dgrad(g.reshape((1, m, 1, n)), a.reshape((m, k, 1, 1)), None, (1, n), *_ONE).reshape((k, n))


def add_rowvec(a, v):
    """a + v with ``v`` broadcast over the leading dimensions of ``a``."""
    _f32(a, v)
    c = v.size
    out = hiparray.empty(a.shape)
    _hip.call('tt_add_rowvec_f32', a.ptr, v.ptr, out.ptr, a.size // c, c)
    return out


def sum_rows(g, c):
    """Sum over all but the trailing ``c`` elements: the gradient of a broadcast bias."""
    _f32(g)
    out = hiparray.empty((c,))
    _hip.call('tt_channel_sum_f32', g.ptr, out.ptr, g.size // c, c, 1)
    return out


def log_softmax_fwd(x):
    _f32(x)
    c = x.shape[-1]
    y = hiparray.empty(x.shape)
    _hip.call('tt_log_softmax_fwd_f32', x.ptr, y.ptr, x.size // c, c)
    return y


def log_softmax_bwd(g, y):
    _f32(g, y)
    c = y.shape[-1]
    dx = hiparray.empty(y.shape)
    _hip.call('tt_log_softmax_bwd_f32', g.ptr, y.ptr, dx.ptr, y.size // c, c)
    return dx


_REDUCTIONS = {'none': 0, 'sum': 1, 'mean': 2}


def _nll_args(logp, target, weight, reduction):
    _f32(logp, weight)
    if logp.ndim != 2 or target.shape != logp.shape[:1]:
        raise RuntimeError(f'the device nll_loss takes logp [N, C] and target [N], got {logp.shape} and {target.shape}')
    if target.dtype != np.int64:
        raise RuntimeError(f'expected an int64 target, got {target.dtype}')
    if reduction not in _REDUCTIONS:
        raise ValueError(f'{reduction} is not a valid value for reduction')
    return _REDUCTIONS[reduction]


def nll_loss_fwd(logp, target, weight, ignore_index, reduction):
    """(loss, count): grad_nn.py:287-327; ``count`` is the device-resident divisor of the mean."""
    red = _nll_args(logp, target, weight, reduction)
    r, c = logp.shape
    out = hiparray.empty((r,) if red == 0 else ())
    count = hiparray.empty((1,))
    _hip.call('tt_nll_loss_fwd_f32', logp.ptr, target.ptr, _ptr(weight), out.ptr, count.ptr, r, c,
              int(ignore_index), red)
    return out, count


def nll_loss_bwd(g, logp_shape, target, weight, count, ignore_index, reduction):
    """grad_nn.py:329-349."""
    _f32(g, weight)
    r, c = logp_shape
    dlogp = hiparray.empty(logp_shape)
    _hip.call('tt_nll_loss_bwd_f32', g.ptr, target.ptr, _ptr(weight), count.ptr, dlogp.ptr, r, c,
              int(ignore_index), _REDUCTIONS[reduction])
    return dlogp
