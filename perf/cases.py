"""Cases that the backend's speed is measured on: the work deepnet has the matrix and conv libraries do,
through their Python entry points.

A case is a dict of plain values; ``prepare`` makes what a training program holds before the call (device
matrices, a net, a seeded generator), ``run`` is one pass.  Matrices live in the library's own device memory
and are filled and handed out as torch tensors over the same memory (no copy).  A pass ends with
``cm.launch_deferred()``: calls that the library holds back to launch together belong to the pass.

  rbm     a contrastive-divergence step through the reference's calls (cudamat/examples/rbm_cudamat.py:46-89 with
          plain updates): propagation up, sample, down, up, statistics
  mlp     NeuralNet.TrainOneBatch of a two-hidden-layer classifier with dropout (deepnet/neuralnet.py:138-337)
  convnet NeuralNet.TrainOneBatch of the net of deepnet/examples/convnet (two conv + pool stages, a dense layer, softmax)
  stage   one conv stage of an edge, forward, backward and weight gradient (deepnet/convolutions.py:5-184)
  conv    the three passes of a convolution layer: convUp, convDown, convOutp
  local   the same three passes of a locally connected layer (one filter bank per module)
  dense   the three products of a fully connected layer: forward, input gradient, accumulated weight gradient
  matrix  the elementwise, broadcast, reduction, softmax and sampling calls on one matrix
"""
import ctypes
import sys
import types

import numpy as np
import torch

from deepnet_amd import convolutions as dc
from deepnet_amd import cudamat as cm
from deepnet_amd import cudamat_conv as cc
from deepnet_amd import layer as dl
from deepnet_amd import neuralnet as dnn
from deepnet_amd import parameter as dp

# ------------------------------------------------------------------ the cases


def listed():
    return [
        # the smallest step in use: MNIST-sized binary RBM, batch 100; a handful of launches
        dict(name='rbm_784x500_b100', kind='rbm', visible=784, hidden=500, batch=100),
        # a wider RBM with sides and a batch that no tile divides
        dict(name='rbm_2001x1003_b250', kind='rbm', visible=2001, hidden=1003, batch=250),
        # the feed-forward classifier of the benchmark, driven by the layer / edge classes
        dict(name='mlp_784_1024_1024_10_b128', kind='mlp', inputs=784, hidden1=1024, hidden2=1024, classes=10, batch=128),
        # deepnet's convnet example at its own batch size of 100, which is no multiple of 16 images
        dict(name='convnet_28_64f5_b100', kind='convnet', side=28, filters=64, hidden=1024, batch=100),
        # first stage of a CIFAR net: conv, max pool, response norm and their gradients
        dict(name='stage_3x32x32_64f5_b128', kind='stage', colors=3, side=32, filters=64, size=5, pool=3, norm=5, batch=128),
        # first layer of an ImageNet net: few colours, large filters, stride
        dict(name='conv_3x224_96f11s4_b128', kind='conv', colors=3, side=224, filters=96, size=11, stride=4, padding=0,
             groups=1, batch=128),
        # second layer of the same net: many colours, two groups
        dict(name='conv_96x27_256f5g2_b128', kind='conv', colors=96, side=27, filters=256, size=5, stride=1, padding=2,
             groups=2, batch=128),
        # locally connected layer on a small map: every module reads its own filter bank
        dict(name='local_64x8_64f3_b128', kind='local', colors=64, side=8, filters=64, size=3, stride=1, padding=1,
             groups=1, batch=128),
        # a large dense layer: as many operations as a call has here
        dict(name='dense_4096x4096_b4096', kind='dense', inputs=4096, outputs=4096, batch=4096),
        # an ordinary one with odd sides
        dict(name='dense_1001x1500_b300', kind='dense', inputs=1001, outputs=1500, batch=300),
        # the 4096 x 4096 op list of the benchmark: streams from memory
        dict(name='matrix_4096x4096', kind='matrix', rows=4096, cols=4096),
        # the same calls on columns that start at any 4-byte boundary
        dict(name='matrix_1001x2047', kind='matrix', rows=1001, cols=2047),
    ]


def _log(rng, lo, hi):
    """A whole number, spread evenly over the logarithm of [lo, hi]."""
    return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))


def _batch(rng):
    """Batches in use: 100 (deepnet's examples), 128 (the benchmark), other whole groups of 16, anything."""
    return rng.choice([100, 128, 16 * rng.randint(2, 16), rng.randint(20, 256)])


def _draw_conv(rng):
    # no more work than the largest listed convolution, 57 GFLOP a pass
    while True:
        first = rng.random() < 0.4
        c = dict(kind='conv', colors=rng.choice([1, 3]) if first else 4 * _log(rng, 4, 48),
                 side=_log(rng, 16, 224) if first else _log(rng, 6, 32), filters=0, size=rng.choice([3, 5, 7]), stride=1,
                 padding=0, groups=1, batch=_batch(rng))
        if first and c['side'] >= 96:
            c['size'], c['stride'] = rng.choice([7, 11]), rng.choice([2, 4])
        elif rng.random() < 0.2:
            c['stride'] = 2
        c['padding'] = rng.choice([0, c['size'] // 2])
        c['filters'] = rng.choice([16 * _log(rng, 1, 16), 16 * _log(rng, 1, 16), _log(rng, 10, 256)])
        if not first and c['filters'] % 32 == 0 and rng.random() < 0.3:
            c['groups'] = 2
        if c['size'] <= c['side'] and _conv_flops(c) <= 57.4e9:
            return c


def draw(rng):
    kind = rng.choice(['rbm', 'mlp', 'convnet', 'stage', 'conv', 'local', 'dense', 'matrix'])
    if kind == 'rbm':
        return dict(kind=kind, visible=_log(rng, 200, 4000), hidden=_log(rng, 100, 2000), batch=_log(rng, 20, 500))
    if kind == 'mlp':
        return dict(kind=kind, inputs=_log(rng, 100, 3000), hidden1=_log(rng, 100, 2048), hidden2=_log(rng, 100, 2048),
                    classes=_log(rng, 5, 200), batch=_log(rng, 32, 512))
    if kind == 'convnet':
        return dict(kind=kind, side=rng.randint(20, 36), filters=16 * rng.randint(2, 6), hidden=_log(rng, 128, 2048),
                    batch=_batch(rng))
    if kind == 'stage':
        return dict(kind=kind, colors=rng.choice([1, 3, 3, 16 * rng.randint(1, 4)]), side=rng.randint(12, 40),
                    filters=16 * rng.randint(1, 6), size=rng.choice([3, 5]), pool=rng.choice([2, 3]),
                    norm=rng.choice([0, 3, 5]), batch=_batch(rng))
    if kind == 'conv':
        return _draw_conv(rng)
    if kind == 'local':
        return dict(kind=kind, colors=4 * rng.randint(2, 24), side=rng.randint(5, 14), filters=16 * rng.randint(1, 6),
                    size=3, stride=1, padding=rng.choice([0, 1]), groups=1, batch=_batch(rng))
    if kind == 'dense':
        return dict(kind=kind, inputs=_log(rng, 64, 4096), outputs=_log(rng, 64, 4096), batch=_log(rng, 32, 4096))
    return dict(kind=kind, rows=_log(rng, 64, 4096), cols=_log(rng, 64, 4096))


# ------------------------------------------------------------------ matrices and tensors


class _Held(object):
    """The device memory of a matrix as torch sees it; given back when no tensor is left that views it."""

    def __init__(self, mat):
        rows, cols = mat.shape
        address = ctypes.cast(mat.mat.data_device, ctypes.c_void_p).value
        self.mat = mat
        self.__cuda_array_interface__ = dict(shape=(cols, rows), typestr='<f4', data=(address, False), version=2)

    def __del__(self):
        if sys is not None and not sys.is_finalizing():
            self.mat.free_device_memory()


def _tensor(mat):
    """A (cols, rows) tensor over the column-major memory of ``mat``, which then belongs to the tensor."""
    return torch.as_tensor(_Held(mat), device='cuda')


class _State(object):
    """What a program holds: ``m`` matrices and ``t`` their tensors by name, besides plain attributes."""

    def __init__(self, case, seed):
        self.case, self.kind, self.m, self.t = case, case['kind'], {}, {}
        self.gen = torch.Generator(device='cuda')
        self.gen.manual_seed(seed)
        cm.CUDAMatrix.init_random(seed % 100003 + 1)     # this program's generator of uniform variates
        self.rnd = (cm.CUDAMatrix.rnd_state, cm.CUDAMatrix.rnd_state_p)

    def new(self, name, rows, cols):
        self.m[name] = cm.empty((rows, cols))
        self.t[name] = _tensor(self.m[name])
        return self.t[name]

    def normal(self, name, rows, cols, scale=1.0):
        self.new(name, rows, cols).normal_(0.0, scale, generator=self.gen)

    def uniform(self, name, rows, cols):
        self.new(name, rows, cols).uniform_(0.0, 1.0, generator=self.gen)

    def classes(self, name, count, cols):
        self.new(name, 1, cols).copy_(torch.randint(0, count, (cols, 1), generator=self.gen, device='cuda'))

    def zeros(self, name, rows, cols):
        self.new(name, rows, cols).zero_()


def _modules(case):
    return (case['side'] + 2 * case['padding'] - case['size']) // case['stride'] + 1


def _conv_flops(case):
    return 2.0 * case['batch'] * case['filters'] * _modules(case) ** 2 * (case['colors'] // case['groups']) * case['size'] ** 2


# ------------------------------------------------------------------ what a program has in hand


def _prepare_rbm(s, c):
    nv, nh, batch = c['visible'], c['hidden'], c['batch']
    s.new('v', nv, batch).copy_(torch.rand((batch, nv), generator=s.gen, device='cuda') < 0.13)
    s.normal('w', nv, nh, 0.01)
    s.normal('bv', nv, 1, 0.1)
    s.normal('bh', nh, 1, 0.1)
    for name in ('h', 'hs', 'h2'):
        s.new(name, nh, batch)
    s.new('v2', nv, batch)


def _run_rbm(s):
    m, eps = s.m, 0.01 / s.case['batch']
    w, v, h, hs, v2, h2, bv, bh = (m[k] for k in ('w', 'v', 'h', 'hs', 'v2', 'h2', 'bv', 'bh'))
    cm.dot(w.T, v, target=h); h.add_col_vec(bh); h.apply_sigmoid()
    h.sample_bernoulli(target=hs)
    cm.dot(w, hs, target=v2); v2.add_col_vec(bv); v2.apply_sigmoid()
    cm.dot(w.T, v2, target=h2); h2.add_col_vec(bh); h2.apply_sigmoid()
    w.add_dot(v, h.T, mult=eps); w.add_dot(v2, h2.T, mult=-eps)
    bv.add_sums(v, axis=1, mult=eps); bv.add_sums(v2, axis=1, mult=-eps)
    bh.add_sums(h, axis=1, mult=eps); bh.add_sums(h2, axis=1, mult=-eps)
    return [s.t[k] for k in ('w', 'bv', 'bh', 'h', 'v2', 'h2')]


def _finish_net(s, net, data):
    """Hands the parameters and the batch of a net over to tensors and keeps what a training loop keeps."""
    s.net, s.step = net, 0
    s.params = []
    for obj in [layer for layer in net.layer if not layer.is_input] + net.edge:
        for key in sorted(obj.params):
            t = _tensor(obj.params[key])
            if obj in net.layer:
                t.normal_(0.0, 0.1, generator=s.gen)      # biases of a net that has been trained for a while
            s.params.append(t)
    for layer, name in data:
        layer.SetData(s.m[name])


def _sgd(**kw):
    return dp.Hyperparams(base_epsilon=0.01, initial_momentum=0.9, final_momentum=0.9, **kw)


def _weights(rng, rows, cols, scale):
    return scale * rng.standard_normal((rows, cols), dtype=np.float32)


def _prepare_mlp(s, c, seed):
    rng, batch = np.random.default_rng(seed), c['batch']
    sizes = (c['inputs'], c['hidden1'], c['hidden2'], c['classes'])
    layers = [dl.LinearLayer('input', sizes[0], batch, hyperparams=dp.Hyperparams(), is_input=True)]
    for i in (1, 2):
        layers.append(dl.ReluLayer('hidden%d' % i, sizes[i], batch, hyperparams=_sgd(activation=dp.RECTIFIED_LINEAR, dropout=True)))
    layers.append(dl.SoftmaxLayer('output', 1, batch, hyperparams=_sgd(activation=dp.SOFTMAX), numlabels=sizes[3], is_output=True,
                                  loss_function=dp.CROSS_ENTROPY))
    edges = [dnn.Edge(layers[i], layers[i + 1], _weights(rng, sizes[i], sizes[i + 1], 0.03), hyperparams=_sgd()) for i in range(3)]
    s.uniform('x', sizes[0], batch)
    s.classes('labels', sizes[3], batch)
    _finish_net(s, dnn.NeuralNet(layers, edges), [(layers[0], 'x'), (layers[-1], 'labels')])


def _prepare_convnet(s, c, seed):
    rng, batch, side, f = np.random.default_rng(seed), c['batch'], c['side'], c['filters']
    s1 = (side - 3) // 2 + 1
    s2 = (s1 - 3) // 2 + 1
    relu = lambda name, dims: dl.ReluLayer(name, dims, batch, hyperparams=_sgd(activation=dp.RECTIFIED_LINEAR))
    layers = [dl.LinearLayer('input_layer', side * side, batch, hyperparams=dp.Hyperparams(), is_input=True),
              relu('hidden1', f * s1 * s1), relu('hidden2', f * s2 * s2), relu('hidden3', c['hidden']),
              dl.SoftmaxLayer('output_layer', 1, batch, hyperparams=_sgd(activation=dp.SOFTMAX), numlabels=10, is_output=True,
                              loss_function=dp.CROSS_ENTROPY)]
    conv = lambda colors: dc.ConvParams(size=5, stride=1, padding=2, num_filters=f, num_colors=colors, max_pool=True, pool_size=3,
                                        pool_stride=2)
    dense = lambda: _sgd(apply_l2_decay=True, l2_decay=0.001)
    edges = [dnn.Edge(layers[0], layers[1], _weights(rng, f, 25, 0.1), hyperparams=_sgd(), conv_params=conv(1)),
             dnn.Edge(layers[1], layers[2], _weights(rng, f, 25 * f, 0.02), hyperparams=_sgd(), conv_params=conv(f)),
             dnn.Edge(layers[2], layers[3], _weights(rng, f * s2 * s2, c['hidden'], 0.02), hyperparams=dense()),
             dnn.Edge(layers[3], layers[4], _weights(rng, c['hidden'], 10, 0.05), hyperparams=dense())]
    s.uniform('x', side * side, batch)
    s.classes('labels', 10, batch)
    _finish_net(s, dnn.NeuralNet(layers, edges), [(layers[0], 'x'), (layers[-1], 'labels')])


def _run_net(s):
    losses = s.net.TrainOneBatch(s.step)
    s.step += 1
    return s.params + [loss.cross_entropy for loss in losses]


def _pooled(c):
    return (c['side'] - c['pool']) // 2 + 1       # the padding keeps the side, pools move by two


def _prepare_stage(s, c):
    n, f, side, pooled = c['batch'], c['filters'], c['side'], _pooled(c)
    params = dc.ConvParams(size=c['size'], stride=1, padding=c['size'] // 2, num_filters=f, num_colors=c['colors'], max_pool=True,
                           pool_size=c['pool'], pool_stride=2, rnorm=c['norm'] > 0, norm_size=c['norm'])
    s.normal('w', f, c['colors'] * c['size'] ** 2, 0.05)
    s.normal('inputs', c['colors'] * side * side, n)
    s.normal('deriv', f * pooled * pooled, n)
    s.new('state', f * pooled * pooled, n)
    s.new('grad', f, c['colors'] * c['size'] ** 2)
    s.new('down', c['colors'] * side * side, n)
    s.edge = dc.ConvEdge(s.m['w'], params, s.m['inputs'].shape, s.m['state'].shape)
    s.keep = [_tensor(b) for b in s.edge.buffers()]
    s.layer = types.SimpleNamespace(dirty=False, is_input=False, deriv=s.m['down'])


def _run_stage(s):
    s.layer.dirty = False
    dc.ConvolveUp(s.m['inputs'], s.edge, s.m['state'])
    dc.AccumulateConvDeriv(s.layer, s.edge, s.m['deriv'])
    dc.ConvOuter(s.edge, s.m['grad'])
    return [s.t[k] for k in ('state', 'down', 'grad')]


def _prepare_conv(s, c, banks=1):
    n, mods = c['batch'], _modules(c)
    taps = banks * (c['colors'] // c['groups']) * c['size'] ** 2
    s.normal('x', n, c['colors'] * c['side'] ** 2)
    s.normal('w', c['filters'], taps, 0.01)
    s.normal('dy', n, c['filters'] * mods * mods)
    s.new('y', n, c['filters'] * mods * mods)
    s.new('dx', n, c['colors'] * c['side'] ** 2)
    s.new('dw', c['filters'], taps)


def _run_conv(s):
    m, c = s.m, s.case
    up, down, outp = (cc.localUp, cc.localDown, cc.localOutp) if s.kind == 'local' else (cc.convUp, cc.convDown, cc.convOutp)
    mods, pad, stride, size, colors, g = _modules(c), c['padding'], c['stride'], c['size'], c['colors'], c['groups']
    up(m['x'], m['w'], m['y'], mods, pad, stride, colors, g)
    down(m['dy'], m['w'], m['dx'], mods, pad, stride, size, c['side'], colors, g)
    outp(m['x'], m['dy'], m['dw'], mods, pad, size, stride, colors, g)
    return [s.t[k] for k in ('y', 'dx', 'dw')]


def _prepare_dense(s, c):
    s.normal('x', c['inputs'], c['batch'])
    s.normal('w', c['inputs'], c['outputs'], 0.03)
    s.normal('dy', c['outputs'], c['batch'])
    s.new('y', c['outputs'], c['batch'])
    s.new('dx', c['inputs'], c['batch'])
    s.zeros('dw', c['inputs'], c['outputs'])


def _run_dense(s):
    m = s.m
    cm.dot(m['w'].T, m['x'], target=m['y'])
    cm.dot(m['w'], m['dy'], target=m['dx'])
    m['dw'].add_dot(m['x'], m['dy'].T, mult=1.0 / s.case['batch'])
    return [s.t[k] for k in ('y', 'dx', 'dw')]


def _prepare_matrix(s, c):
    rows, cols = c['rows'], c['cols']
    s.normal('a', rows, cols, 2.0)           # inputs of units
    s.normal('b', rows, cols)
    s.uniform('p', rows, cols)
    s.zeros('acc', rows, cols)
    s.normal('col', rows, 1)
    s.normal('row', 1, cols)
    for name in ('mult', 'sigmoid', 'exp', 'by_col', 'plus_row', 'softmax', 'rand', 'sample'):
        s.new(name, rows, cols)
    for name in ('sum0', 'max0'):
        s.new(name, 1, cols)
    for name in ('sum1', 'max1'):
        s.new(name, rows, 1)


def _run_matrix(s):
    m, a = s.m, s.m['a']
    m['acc'].add_mult(m['b'], 0.5)
    a.mult(m['b'], target=m['mult'])
    a.apply_sigmoid(target=m['sigmoid'])
    cm.exp(a, target=m['exp'])
    a.mult_by_col(m['col'], target=m['by_col'])
    a.add_row_vec(m['row'], target=m['plus_row'])
    a.sum(axis=0, target=m['sum0'])
    a.sum(axis=1, target=m['sum1'])
    a.max(axis=0, target=m['max0'])
    a.max(axis=1, target=m['max1'])
    a.apply_softmax(target=m['softmax'])
    m['rand'].fill_with_rand()
    m['p'].sample_bernoulli(target=m['sample'])
    return [s.t[k] for k in ('acc', 'mult', 'sigmoid', 'exp', 'by_col', 'plus_row', 'sum0', 'sum1', 'max0', 'max1', 'softmax',
                             'rand', 'sample')]


def prepare(case, seed):
    s = _State(case, seed)
    kind = s.kind
    if kind == 'rbm':
        _prepare_rbm(s, case)
    elif kind == 'mlp':
        _prepare_mlp(s, case, seed)
    elif kind == 'convnet':
        _prepare_convnet(s, case, seed)
    elif kind == 'stage':
        _prepare_stage(s, case)
    elif kind == 'conv':
        _prepare_conv(s, case)
    elif kind == 'local':
        _prepare_conv(s, case, banks=_modules(case) ** 2)
    elif kind == 'dense':
        _prepare_dense(s, case)
    else:
        _prepare_matrix(s, case)
    return s


_RUN = dict(rbm=_run_rbm, mlp=_run_net, convnet=_run_net, stage=_run_stage, conv=_run_conv, local=_run_conv, dense=_run_dense,
            matrix=_run_matrix)


def run(state):
    cm.CUDAMatrix.rnd_state, cm.CUDAMatrix.rnd_state_p = state.rnd
    out = _RUN[state.kind](state)
    cm.launch_deferred()
    return out


# ------------------------------------------------------------------ what a pass cannot do without


def work(case):
    """Floating-point operations of the products, and 4 bytes for every element read first or written last."""
    c, kind = case, case['kind']
    n = c.get('batch', 0)
    if kind == 'rbm':
        nv, nh = c['visible'], c['hidden']
        return dict(flops=10.0 * nv * nh * n, bytes=4.0 * (2 * nv * nh + 2 * (nv + nh) + 2 * nv * n + 3 * nh * n))
    if kind == 'mlp':
        dims = (c['inputs'], c['hidden1'], c['hidden2'], c['classes'])
        params = [dims[i] * dims[i + 1] for i in range(3)]
        # the first layer needs no input gradient; weight and momentum are read and written; states, masks, gradients once
        return dict(flops=2.0 * n * (3 * sum(params) - params[0]),
                    bytes=4.0 * (4 * sum(params) + n * (dims[0] + 3 * dims[1] + 3 * dims[2] + 2 * dims[3])))
    if kind == 'convnet':
        side, f = c['side'], c['filters']
        s1 = (side - 3) // 2 + 1
        s2 = (s1 - 3) // 2 + 1
        conv1, conv2 = 25.0 * f * side * side, 25.0 * f * f * s1 * s1
        params = f * s2 * s2 * c['hidden'] + c['hidden'] * 10
        maps = 2 * f * (side * side + 2 * s1 * s1 + s2 * s2) + side * side + 2 * c['hidden']
        return dict(flops=2.0 * n * (2 * conv1 + 3 * conv2 + 3 * params), bytes=4.0 * (4 * (params + 25 * f + 25 * f * f) + n * maps))
    if kind == 'stage':
        pooled = _pooled(c)
        taps = c['colors'] * c['size'] ** 2
        image, up, out = c['colors'] * c['side'] ** 2, c['filters'] * c['side'] ** 2, c['filters'] * pooled ** 2
        # inputs, activations before and after pooling, the output gradient and both gradients on the way down
        return dict(flops=6.0 * n * up * taps, bytes=4.0 * (2 * c['filters'] * taps + n * (2 * image + 2 * up + 3 * out)))
    if kind in ('conv', 'local'):
        mods = _modules(c) ** 2
        taps = (mods if kind == 'local' else 1) * (c['colors'] // c['groups']) * c['size'] ** 2
        return dict(flops=3 * _conv_flops(c),
                    bytes=4.0 * (2 * n * c['colors'] * c['side'] ** 2 + 2 * n * c['filters'] * mods + 2 * c['filters'] * taps))
    if kind == 'dense':
        i, o = c['inputs'], c['outputs']
        return dict(flops=6.0 * i * o * n, bytes=4.0 * (2 * i * n + 2 * o * n + 3 * i * o))
    e = c['rows'] * c['cols']
    # a, b, p and acc are read once, nine matrices are written
    return dict(flops=20.0 * e, bytes=4.0 * (13 * e + 3 * (c['rows'] + c['cols'])))


def tolerance(case):
    """About four times what was seen against 64-bit sums (conv, dense, matrix) and with weights moved by their last bit."""
    kind = case['kind']
    if kind == 'rbm':
        # A uniform draw that falls between two roundings of a unit's probability flips its sample (about one unit in
        # 10^7), and one flip moves the reconstruction of one case of the batch: 2e-4 of the whole at batch 100.
        return dict(rel=2e-3, max=0.05)
    if kind == 'mlp':
        return dict(rel=2e-6, max=1e-4)
    # Two candidates of a pooling window that are equal to rounding exchange their roles in the gradient (about one
    # window in 10^6 or 10^7): one gradient value moves by a pixel.
    if kind == 'convnet':
        return dict(rel=2e-5, max=1e-3)
    if kind == 'stage':
        return dict(rel=4e-3, max=0.5)
    if kind in ('conv', 'local', 'dense'):
        return dict(rel=5e-6, max=5e-5)
    return dict(rel=1e-6, max=4e-6)
