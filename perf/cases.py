"""The work this framework is timed on: what its users run, through the public entry points.

Four kinds of case.  ``classifier`` and ``generator`` / ``discriminator`` are whole networks of the
reference's examples (ResNet-50 finetuning at 224x224, PreAct-ResNet-18 on 32x32 images, the two
halves of the 64x64 DCGAN): a training step -- forward, loss, backward, optimiser -- or an evaluation
pass.  ``conv``, ``norm`` and ``pool`` are single layers called as a user's own network calls them,
forward and backward, in sizes that need not fit any tile.  Three convolution arithmetics are offered
to the user (``tt.cuda.set_conv_math``) and all three are in use: float32 (the default), bfloat16
operands, and float32 carried out in three bfloat16 terms.

``listed()`` are fixed cases, ``draw(rng)`` makes others of the same ranges.  Device arrays come back
as torch tensors on the same memory (no copy, no synchronisation).
"""
import math

import numpy as np
import torch

import pytortto_amd as tt
from pytortto_amd import nn
from pytortto_amd.xparray import hiparray

F = nn.functional


# ---- the cases -------------------------------------------------------------------------------------

def _conv(name, n, c, h, w, k, r, s, stride=(1, 1), pad=(0, 0), dil=(1, 1), groups=1, bias=False, transposed=False,
          math='f32'):
    case = {'kind': 'conv', 'n': n, 'c': c, 'h': h, 'w': w, 'k': k, 'r': r, 's': s, 'sh': stride[0], 'sw': stride[1],
            'ph': pad[0], 'pw': pad[1], 'dh': dil[0], 'dw': dil[1], 'groups': groups, 'bias': bias,
            'transposed': transposed, 'math': math}
    return dict(case, name=name) if name else case


def listed():
    return [
        # the flagship: a ResNet-50 training step at the benchmark's batch, default arithmetic
        {'name': 'resnet50_train_b64_f32', 'kind': 'classifier', 'net': 'resnet50', 'train': True, 'batch': 64,
         'size': 224, 'math': 'f32'},
        # the same network as the finetuning example runs it (batch 32), with bf16 arithmetic for speed
        {'name': 'resnet50_train_b32_bf16', 'kind': 'classifier', 'net': 'resnet50', 'train': True, 'batch': 32,
         'size': 224, 'math': 'bf16'},
        # a pair of images through the finished network: latency and launches count, not throughput
        {'name': 'resnet50_eval_b2_f32', 'kind': 'classifier', 'net': 'resnet50', 'train': False, 'batch': 2,
         'size': 224, 'math': 'f32'},
        # the validation loop over a whole set: forward only, large batches
        {'name': 'resnet50_eval_b64_bf16', 'kind': 'classifier', 'net': 'resnet50', 'train': False, 'batch': 64,
         'size': 224, 'math': 'bf16'},
        # the CIFAR-10 example at its own batch, default arithmetic and the faster float32 one
        {'name': 'preact18_train_b128_f32', 'kind': 'classifier', 'net': 'preact18', 'train': True, 'batch': 128,
         'size': 32, 'math': 'f32'},
        {'name': 'preact18_train_b128_bf16x3', 'kind': 'classifier', 'net': 'preact18', 'train': True, 'batch': 128,
         'size': 32, 'math': 'bf16x3'},
        # the transposed convolutions: the generator of the DCGAN example at its batch, Adam
        {'name': 'dcgan_generator_b128_f32', 'kind': 'generator', 'batch': 128, 'width': 64, 'math': 'f32'},
        # the smallest layer anybody times: Conv2d(16, 32, 3, padding=1) on [32,16,32,32], with bias
        _conv('conv_small_3x3_f32', 32, 16, 32, 32, 32, 3, 3, pad=(1, 1), bias=True),
        # the geometry of the reference's own speed notebook: groups, unequal strides, dilation, odd sizes
        _conv('conv_grouped_odd_f32', 128, 4, 64, 64, 16, 3, 2, stride=(1, 3), pad=(2, 3), dil=(1, 2), groups=2,
              bias=True),
        # a mid-network 3x3 layer on an image that fits no tile
        _conv('conv_ragged_3x3_bf16x3', 24, 160, 45, 37, 192, 3, 3, pad=(1, 1), math='bf16x3'),
        # BatchNorm with the ReLU behind it at the size of a first-stage output
        {'name': 'norm_relu_256x56x56', 'kind': 'norm', 'n': 64, 'c': 256, 'h': 56, 'w': 56, 'relu': True},
        # the pooling behind the stem
        {'name': 'pool_64x112x112', 'kind': 'pool', 'n': 64, 'c': 64, 'h': 112, 'w': 112, 'k': 3, 'stride': 2, 'pad': 1},
    ]


def _spread(rng, lo, hi):
    """A whole number between lo and hi, even over the logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _draw_conv(rng, math_mode):
    transposed = rng.random() < 0.25
    groups = rng.choice((1, 1, 1, 1, 2, 4))
    r, s = rng.choice(((1, 1), (1, 1), (3, 3), (3, 3), (3, 3), (3, 3), (5, 5), (4, 4), (3, 2), (7, 7)))
    stride = rng.choice(((1, 1), (1, 1), (2, 2), (2, 2), (1, 3))) if (r, s) != (7, 7) else (2, 2)
    dil = rng.choice(((1, 1), (1, 1), (1, 1), (2, 2), (1, 2))) if r == 3 else (1, 1)
    pad = rng.choice(((r // 2, s // 2), (r // 2, s // 2), (0, 0)))
    while True:
        n = _spread(rng, 1, 160)
        c, k = groups * _spread(rng, 2, 640), groups * _spread(rng, 3, 640)
        h, w = _spread(rng, 7, 128), _spread(rng, 7, 128)
        case = _conv(None, n, c, h, w, k, r, s, stride, pad, dil, groups, rng.random() < 0.4, transposed, math_mode)
        p, q = _out_hw(case)
        if p > 0 and q > 0 and work(case)['flops'] < 4e11 and n * max(c * h * w, k * p * q) < 1 << 26:
            return case


def draw(rng):
    kind = rng.choice(('classifier', 'classifier', 'gan', 'conv', 'conv', 'conv', 'norm', 'pool'))
    mode = rng.choice(('f32', 'f32', 'f32', 'bf16', 'bf16x3'))
    if kind == 'classifier':
        train = rng.random() < 0.6
        if rng.random() < 0.5:
            return {'kind': 'classifier', 'net': 'resnet50', 'train': train, 'batch': _spread(rng, 8 if train else 2, 60),
                    'size': rng.choice((160, 176, 192, 200, 224)), 'math': mode}
        return {'kind': 'classifier', 'net': 'preact18', 'train': train, 'batch': _spread(rng, 16 if train else 2, 250),
                'size': rng.choice((28, 32, 36, 40)), 'math': mode}
    if kind == 'gan':
        return {'kind': rng.choice(('generator', 'discriminator')), 'batch': _spread(rng, 8, 200),
                'width': rng.choice((32, 48, 64, 96)), 'math': mode}
    if kind == 'conv':
        return _draw_conv(rng, mode)
    while True:
        n, c, h, w = _spread(rng, 1, 256), _spread(rng, 3, 1024), _spread(rng, 4, 160), _spread(rng, 4, 160)
        if 1 << 13 <= n * c * h * w <= 1 << 26:
            break
    if kind == 'norm':
        return {'kind': 'norm', 'n': n, 'c': c, 'h': h, 'w': w, 'relu': rng.random() < 0.6}
    k, stride, pad = rng.choice(((3, 2, 1), (3, 2, 1), (2, 2, 0), (3, 1, 1)))
    return {'kind': 'pool', 'n': n, 'c': c, 'h': h, 'w': w, 'k': k, 'stride': stride, 'pad': pad}


# ---- the networks of the examples ------------------------------------------------------------------

def _conv1x1(cin, cout, stride=1):
    return nn.Conv2d(cin, cout, kernel_size=1, stride=stride, bias=False)


def _conv3x3(cin, cout, stride=1):
    return nn.Conv2d(cin, cout, kernel_size=3, stride=stride, padding=1, bias=False)


class Bottleneck(nn.Module):
    def __init__(self, cin, width, stride, downsample):
        super().__init__()
        self.conv1, self.bn1 = _conv1x1(cin, width), nn.BatchNorm2d(width)
        self.conv2, self.bn2 = _conv3x3(width, width, stride), nn.BatchNorm2d(width)
        self.conv3, self.bn3 = _conv1x1(width, width * 4), nn.BatchNorm2d(width * 4)
        self.downsample = downsample

    def forward(self, x):
        shortcut = x if self.downsample is None else self.downsample(x)
        out = F.relu(self.bn1(self.conv1(x)))
        out = F.relu(self.bn2(self.conv2(out)))
        out = self.bn3(self.conv3(out))
        return F.relu(out + shortcut)


class ResNet50(nn.Module):
    def __init__(self):
        super().__init__()
        self.conv1 = nn.Conv2d(3, 64, kernel_size=7, stride=2, padding=3, bias=False)
        self.bn1 = nn.BatchNorm2d(64)
        self.maxpool = nn.MaxPool2d(kernel_size=3, stride=2, padding=1)
        blocks, cin = [], 64
        for width, count, stride in ((64, 3, 1), (128, 4, 2), (256, 6, 2), (512, 3, 2)):
            for i in range(count):
                down = nn.Sequential(_conv1x1(cin, width * 4, stride), nn.BatchNorm2d(width * 4)) if i == 0 else None
                blocks.append(Bottleneck(cin, width, stride if i == 0 else 1, down))
                cin = width * 4
        self.layers = nn.Sequential(*blocks)
        self.classifier = nn.Linear(2048, 10)

    def forward(self, x):
        x = self.maxpool(F.relu(self.bn1(self.conv1(x))))
        x = self.layers(x)
        x = tt.flatten(tt.mean(x, (-1, -2), True), 1)
        return F.log_softmax(self.classifier(x), -1)


class PreActBlock(nn.Module):
    def __init__(self, cin, cout, stride):
        super().__init__()
        self.bn1, self.conv1 = nn.BatchNorm2d(cin), _conv3x3(cin, cout, stride)
        self.bn2, self.conv2 = nn.BatchNorm2d(cout), _conv3x3(cout, cout)
        self.shortcut = None if stride == 1 and cin == cout else _conv1x1(cin, cout, stride)

    def forward(self, x):
        out = self.conv1(F.relu(self.bn1(x)))
        out = self.conv2(F.relu(self.bn2(out)))
        return out + (x if self.shortcut is None else self.shortcut(x))


class PreActResNet18(nn.Module):
    def __init__(self):
        super().__init__()
        layers, cin = [_conv3x3(3, 64)], 64
        for cout, stride in ((64, 1), (128, 2), (256, 2), (512, 2)):
            layers += [PreActBlock(cin, cout, stride), PreActBlock(cout, cout, 1)]
            cin = cout
        self.layers, self.bn = nn.Sequential(*layers), nn.BatchNorm2d(512)
        self.classifier = nn.Linear(512, 10)

    def forward(self, x):
        x = F.relu(self.bn(self.layers(x)))
        return F.log_softmax(self.classifier(tt.flatten(tt.mean(x, (-1, -2), True), 1)), -1)


def _generator(width):
    layers, cin = [], 100
    for cout, stride, pad in ((8 * width, 1, 0), (4 * width, 2, 1), (2 * width, 2, 1), (width, 2, 1)):
        layers += [nn.ConvTranspose2d(cin, cout, 4, stride, pad, bias=False), nn.BatchNorm2d(cout), nn.ReLU()]
        cin = cout
    return nn.Sequential(*layers, nn.ConvTranspose2d(cin, 3, 4, 2, 1, bias=False))


def _discriminator(width):
    layers = [nn.Conv2d(3, width, 4, 2, 1, bias=False), nn.LeakyReLU(0.2)]
    for i in (1, 2, 4):
        layers += [nn.Conv2d(i * width, 2 * i * width, 4, 2, 1, bias=False), nn.BatchNorm2d(2 * i * width),
                   nn.LeakyReLU(0.2)]
    return nn.Sequential(*layers, nn.Conv2d(8 * width, 1, 4, 1, 0, bias=False))


# ---- device arrays and torch tensors ---------------------------------------------------------------

class _Memory:
    """What torch needs to know to put a tensor on a device array's memory; keeps the array alive."""

    def __init__(self, array):
        self.array = array
        self.__cuda_array_interface__ = {'shape': array.shape, 'typestr': array.dtype.str, 'data': (array.ptr, False),
                                         'strides': None, 'version': 2}


def _torch(array):
    return torch.as_tensor(_Memory(array), device='cuda')


def _normal(gen, shape, mean=0.0, std=1.0):
    """A device tensor of the framework with values drawn on the GPU."""
    array = hiparray.empty(shape)
    _torch(array).copy_(torch.randn(shape, generator=gen, device='cuda') * std + mean)
    return tt.Tensor(array)


def _out_hw(case):
    h, w = case['h'], case['w']
    if case['transposed']:
        return ((h - 1) * case['sh'] - 2 * case['ph'] + case['dh'] * (case['r'] - 1) + 1,
                (w - 1) * case['sw'] - 2 * case['pw'] + case['dw'] * (case['s'] - 1) + 1)
    return ((h + 2 * case['ph'] - case['dh'] * (case['r'] - 1) - 1) // case['sh'] + 1,
            (w + 2 * case['pw'] - case['dw'] * (case['s'] - 1) - 1) // case['sw'] + 1)


def _trained_statistics(net, rng):
    """Running statistics and affine parameters of the size that training leaves: activations of unit
    scale, halved by the ReLU, through weights of variance 1 / (3 fan_in); a residual branch ends in
    factors well below one."""
    last = {id(m.bn3) for m in net.modules() if isinstance(m, Bottleneck)}
    for m in net.modules():
        if isinstance(m, nn.BatchNorm2d):
            c = m.running_mean.shape[0]
            m.running_mean.copy_(rng.normal(0.0, 0.1, c).astype(np.float32))
            m.running_var.copy_(rng.uniform(0.1, 0.3, c).astype(np.float32))
            with tt.no_grad():
                m.weight.copy_((rng.uniform(0.5, 1.2, c) * (0.25 if id(m) in last else 1.0)).astype(np.float32))
                m.bias.copy_(rng.normal(0.0, 0.1, c).astype(np.float32))


def prepare(case, seed):
    tt.manual_seed(seed % (1 << 32))
    gen = torch.Generator('cuda')
    gen.manual_seed(seed)
    state, kind = {'case': case, 'math': case.get('math', 'f32')}, case['kind']
    if kind == 'classifier':
        finetuned = case['net'] == 'resnet50'
        net = ResNet50() if finetuned else PreActResNet18()
        if finetuned or not case['train']:
            _trained_statistics(net, np.random.default_rng(seed))
        if not case['train']:
            net.eval()
        net.cuda()
        state['net'] = net
        state['x'] = _normal(gen, (case['batch'], 3, case['size'], case['size']))
        state['target'] = tt.tensor(np.random.default_rng(seed).integers(0, 10, case['batch'])).cuda()
        state['opt'] = tt.optim.SGD(net.parameters(), lr=0.001 if finetuned else 0.01, momentum=0.9,
                                    weight_decay=5e-4)
        state['returned'] = [m.weight for m in net.modules() if isinstance(m, (nn.Conv2d, nn.Linear))]
    elif kind in ('generator', 'discriminator'):
        b = case['batch']
        net = (_generator if kind == 'generator' else _discriminator)(case['width'])
        net.cuda()
        state['net'] = net
        state['x'] = _normal(gen, (b, 100, 1, 1) if kind == 'generator' else (b, 3, 64, 64))
        # what the loss hands back: small, of either sign
        state['gradient'] = _normal(gen, (b, 3, 64, 64) if kind == 'generator' else (b, 1, 1, 1), std=0.01)
        state['opt'] = tt.optim.Adam(net.parameters(), lr=2e-4, betas=(0.5, 0.999))
        state['returned'] = [m.weight for m in net.modules() if isinstance(m, (nn.Conv2d, nn.ConvTranspose2d))]
    else:
        n, c, h, w = case['n'], case['c'], case['h'], case['w']
        if kind == 'conv':
            make = nn.ConvTranspose2d if case['transposed'] else nn.Conv2d
            layer = make(c, case['k'], (case['r'], case['s']), (case['sh'], case['sw']), (case['ph'], case['pw']),
                         groups=case['groups'], bias=case['bias'], dilation=(case['dh'], case['dw']))
            out = (n, case['k']) + _out_hw(case)
        elif kind == 'norm':
            layer, out = nn.BatchNorm2d(c), (n, c, h, w)
        else:
            layer = nn.MaxPool2d(case['k'], case['stride'], case['pad'])
            out = (n, c) + tuple((v + 2 * case['pad'] - case['k']) // case['stride'] + 1 for v in (h, w))
        layer.cuda()
        state['layer'] = layer
        # activations of a normalised network; BatchNorm sees a convolution's output, off centre
        state['x'] = _normal(gen, (n, c, h, w), *((0.5, 2.0) if kind == 'norm' else ()))
        state['x'].requires_grad = True
        state['gradient'] = _normal(gen, out, std=0.1)
    torch.cuda.synchronize()
    return state


def run(state):
    tt.cuda.set_conv_math(state['math'])
    case = state['case']
    kind = case['kind']
    if kind == 'classifier':
        net = state['net']
        if not case['train']:
            with tt.no_grad():
                return _torch(net(state['x']).data)
        state['opt'].zero_grad()
        logp = net(state['x'])
        loss = F.nll_loss(logp, state['target'])
        loss.backward()
        state['opt'].step()
        return [_torch(loss.data), _torch(logp.data)] + [_torch(p.data) for p in state['returned']]
    if 'net' in state:
        state['opt'].zero_grad()
        y = state['net'](state['x'])
        y.backward(state['gradient'])
        state['opt'].step()
        return [_torch(y.data)] + [_torch(p.data) for p in state['returned']]
    x, layer = state['x'], state['layer']
    x.grad = None
    for p in layer.parameters():
        p.grad = None
    y = layer(x)
    if case.get('relu'):
        y = F.relu(y)
    y.backward(state['gradient'])
    return [_torch(y.data), _torch(x.grad)] + [_torch(p.grad) for p in layer.parameters()]


# ---- what a pass cannot do without -----------------------------------------------------------------

def _conv_work(n, c, h, w, k, r, s, p, q, groups=1, transposed=False):
    """(multiply-add FLOPs of one pass, output elements, weights)"""
    pixels = h * w if transposed else p * q
    return 2.0 * n * (c // groups) * k * r * s * pixels, n * k * p * q, c * k * r * s // groups


def _net_layers(case):
    b, layers = case['batch'], []
    if case['kind'] == 'classifier':
        def half(v):
            return (v - 1) // 2 + 1
        v = case['size']
        if case['net'] == 'resnet50':
            v = half(v)
            layers.append((b, 3, case['size'], case['size'], 64, 7, 7, v, v))
            v, cin = half(v), 64
            for width, count, stride in ((64, 3, 1), (128, 4, 2), (256, 6, 2), (512, 3, 2)):
                for i in range(count):
                    u = half(v) if i == 0 and stride == 2 else v
                    layers += [(b, cin, v, v, width, 1, 1, v, v), (b, width, v, v, width, 3, 3, u, u),
                               (b, width, u, u, 4 * width, 1, 1, u, u)]
                    if i == 0:
                        layers.append((b, cin, v, v, 4 * width, 1, 1, u, u))
                    v, cin = u, 4 * width
        else:
            layers.append((b, 3, v, v, 64, 3, 3, v, v))
            cin = 64
            for cout, stride in ((64, 1), (128, 2), (256, 2), (512, 2)):
                u = half(v) if stride == 2 else v
                layers += [(b, cin, v, v, cout, 3, 3, u, u), (b, cout, u, u, cout, 3, 3, u, u)]
                if stride == 2:
                    layers.append((b, cin, v, v, cout, 1, 1, u, u))
                layers += [(b, cout, u, u, cout, 3, 3, u, u)] * 2
                v, cin = u, cout
        return [l + (1, False) for l in layers]
    w = case['width']
    if case['kind'] == 'generator':
        return [(b, ci, h, h, co, 4, 4, o, o, 1, True) for ci, h, co, o in
                ((100, 1, 8 * w, 4), (8 * w, 4, 4 * w, 8), (4 * w, 8, 2 * w, 16), (2 * w, 16, w, 32), (w, 32, 3, 64))]
    return [(b, ci, h, h, co, 4, 4, o, o, 1, False) for ci, h, co, o in
            ((3, 64, w, 32), (w, 32, 2 * w, 16), (2 * w, 16, 4 * w, 8), (4 * w, 8, 8 * w, 4), (8 * w, 4, 1, 1))]


def work(case):
    """A network: every convolution's output written once (and, in training, read once by the backward
    pass), weights read once (training: gradient written, weight and optimiser state updated).  A layer:
    x, dy and the weights read once, y, dx and the gradients written once."""
    kind = case['kind']
    if kind in ('classifier', 'generator', 'discriminator'):
        parts = [_conv_work(*l) for l in _net_layers(case)]
        flops, acts, weights = (sum(v) for v in zip(*parts))
        if not case.get('train', True):
            return {'bytes': 4.0 * (acts + weights), 'flops': flops}
        # the first layer's input needs no gradient
        return {'bytes': 4.0 * (2 * acts + (6 if kind == 'classifier' else 8) * weights), 'flops': 3 * flops - parts[0][0]}
    n, c, h, w = case['n'], case['c'], case['h'], case['w']
    if kind == 'conv':
        p, q = _out_hw(case)
        flops, y, weights = _conv_work(n, c, h, w, case['k'], case['r'], case['s'], p, q, case['groups'],
                                       case['transposed'])
        return {'bytes': 4.0 * (2 * n * c * h * w + 2 * y + 2 * weights), 'flops': 3 * flops}
    if kind == 'norm':
        return {'bytes': 16.0 * n * c * h * w, 'flops': 12.0 * n * c * h * w}
    p, q = ((v + 2 * case['pad'] - case['k']) // case['stride'] + 1 for v in (h, w))
    return {'bytes': 8.0 * n * c * (h * w + p * q), 'flops': float(n * c * p * q * case['k'] ** 2)}


def tolerance(case):
    """About four times what two correct evaluations were seen to differ by, over 130 cases of these
    ranges: float32 results between float32 and three-term arithmetic (another order of summation), bf16
    ones against float32 arithmetic, BatchNorm against float64."""
    kind, half = case['kind'], case.get('math') == 'bf16'
    if kind == 'pool':
        return 'exact'                                  # values are copied
    if kind == 'norm':
        return {'rel': 5e-7, 'max': 1e-6}               # seen: 1e-7, 2.3e-7
    if kind == 'conv':
        return {'rel': 1e-2, 'max': 6e-2} if half else {'rel': 7e-6, 'max': 7e-5}       # seen: 2.4e-3; 1.6e-6
    if kind == 'classifier':
        if half:
            return {'rel': 4e-3, 'max': 1.2e-2}         # seen: 1e-3
        return {'rel': 7e-5, 'max': 4e-3} if case['train'] else {'rel': 3e-6, 'max': 6e-6}      # seen: 1.6e-5; 8e-7
    # Adam's first steps move a weight by the sign of its gradient, whatever its size
    return {'rel': 3e-2, 'max': 0.3} if half else {'rel': 4e-3, 'max': 0.3}     # seen: 1e-2; 9e-4
