'''The work that is timed: programs of this package's workloads, over the range of sizes in which they are used.

A case names a program and its sizes and says how a pass is made:

* `call`: a whole call of the wrapped function, `vkjax_amd.wrap(f)(params, x)`: host arrays in, host arrays out, with
  uploads, launches, downloads and the Python around them; the weights are read-only arrays, which stay in HBM by themselves.
  This is how a program serves requests.
* `replay`: one replay of the recorded launches on arguments that already lie in HBM, results left there
  (`JaxprInterpreter.upload_inputs` / `.replay`): the form the throughput of a network is quoted in, and the way a program
  works whose data stay on the device. The outputs are the result arrays in HBM themselves.

A training step returns its loss and the updated weights. Nothing here is specific to one size: `draw` takes the same
programs at sizes spread over the ranges that the listed cases stand for.
'''
import ctypes

import numpy as np
import torch

import vkjax_amd
from vkjax_amd import minijax as mj
from vkjax_amd import workloads as W
from vkjax_amd.jaxpr_interpreter import JaxprInterpreter
from vkjax_amd.minijax import tree_util

jnp, nn = mj.numpy, mj.nn


# ------------------------------------------------------------------ the programs

def softmax_labels(x):
    '''Class probabilities and labels of rows of scores.'''
    p = nn.softmax(x, axis=-1)
    return p, jnp.argmax(p, axis=1)


def normalised_residual(params, x, r):
    '''Inference-mode batch norm, residual addition and ReLU of an activation, and its global average.'''
    y = nn.relu(nn.batch_norm_inference(x, params['scale'], params['shift'], params['mean'], params['var']) + r)
    return y, jnp.mean(y, axis=(1, 2))


def _with_kernels(tree, kernels):
    '''The parameter tree of the network with its convolution kernels and dense layer taken from `kernels` (a flat dict).'''
    def walk(node, path):
        if not isinstance(node, dict):
            return kernels.get(path, node)
        return {k: walk(v, f'{path}/{k}' if path else k) for k, v in node.items()}
    return walk(tree, '')


def _kernels(tree, path=''):
    if not isinstance(tree, dict):
        return {path: tree} if path.endswith('/w') or path == 'fc/b' else {}
    found = {}
    for k, v in tree.items():
        found.update(_kernels(v, f'{path}/{k}' if path else k))
    return found


def resnet50_kernels_step(kernels, params, x, onehot):
    '''One SGD step of ResNet-50 on its convolution kernels and its dense layer with batch norm frozen (the usual way to
    train on from a network whose statistics are to stay): the loss and the updated arrays.'''
    def loss(kernels, params, x, onehot):
        logits, _ = W.resnet50(_with_kernels(params, kernels), x)
        return W.softmax_cross_entropy(logits, onehot)
    value, grads = mj.value_and_grad(loss)(kernels, params, x, onehot)
    return value, {name: kernels[name] - np.float32(0.01) * grads[name] for name in kernels}


def _program(case):
    p = case['program']
    if p == 'rng_uniform':
        shape = (case['rows'], case['cols'])
        return lambda key: W.rng_uniform(key, shape)
    return {'affine': W.affine, 'mlp': W.mlp, 'mlp_train': W.mlp_train_step, 'conv_block': W.conv_block, 'resnet50': W.resnet50,
            'convnet_train': W.convnet_train_step, 'resnet50_train': resnet50_kernels_step, 'gather_scatter': W.gather_scatter,
            'softmax_labels': softmax_labels, 'normalised_residual': normalised_residual}[p]


def _inputs(case, seed):
    '''The program's arguments: uniform images, samples and tables, He-normal weights, as the package's workloads make them.'''
    p = case['program']
    rng = np.random.default_rng(seed)
    if p == 'affine':
        m, k, n = case['batch'], case['features'], case['outputs']
        return [rng.random((m, k), dtype=np.float32), rng.random((k, n), dtype=np.float32), rng.random((n,), dtype=np.float32)]
    if p in ('mlp', 'mlp_train'):
        sizes = (case['features'], case['hidden'], case['hidden2'], case['classes'])
        return (W.mlp_inputs if p == 'mlp' else W.mlp_train_inputs)(seed, case['batch'], sizes)
    if p == 'conv_block':
        return W.conv_block_inputs(seed, case['batch'], case['size'], case['channels'])
    if p == 'convnet_train':
        return W.convnet_train_inputs(seed, case['batch'], case['size'], (3, case['channels'], case['channels2']))
    if p == 'resnet50':
        return W.resnet50_inputs(seed, case['batch'], case['size'])
    if p == 'resnet50_train':
        params, x, onehot = W.resnet50_train_inputs(seed, case['batch'], case['size'])
        return [_kernels(params), params, x, onehot]
    if p == 'rng_uniform':
        return W.rng_inputs(seed)
    if p == 'gather_scatter':
        return W.gather_scatter_inputs(seed, case['rows'], case['cols'], case['lookups'], case['bag'])
    if p == 'softmax_labels':
        return [4.0 * rng.standard_normal((case['rows'], case['cols']), dtype=np.float32)]
    if p == 'normalised_residual':
        c, shape = case['channels'], (case['batch'], case['size'], case['size'], case['channels'])
        bn = dict(scale=(0.5 + rng.random(c, dtype=np.float32)), shift=0.1 * rng.standard_normal(c, dtype=np.float32),
                  mean=0.1 * rng.standard_normal(c, dtype=np.float32), var=(0.5 + rng.random(c, dtype=np.float32)))
        return [bn, rng.standard_normal(shape, dtype=np.float32), rng.standard_normal(shape, dtype=np.float32)]
    raise ValueError(p)


# ------------------------------------------------------------------ the cases

def listed():
    return [
        #the smallest call there is: one dense layer on eight samples; host work and the launch itself
        dict(name='affine_8_call', program='affine', way='call', batch=8, features=128, outputs=16),
        #a classifier that serves batches of samples
        dict(name='mlp_256_call', program='mlp', way='call', batch=256, features=784, hidden=512, hidden2=512, classes=10),
        #a training step of a small dense network, with a last batch that is no round number and odd widths
        dict(name='mlp_train_ragged', program='mlp_train', way='replay', batch=1000, features=784, hidden=300, hidden2=100, classes=10),
        #one convolution block in the middle of a network
        dict(name='conv_block_32', program='conv_block', way='replay', batch=32, size=56, channels=64),
        #a training step of a small convolutional network, odd image size and batch: strided and padded convolutions, max and
        #average pooling, and all their gradients
        dict(name='convnet_train_odd', program='convnet_train', way='replay', batch=50, size=97, channels=64, channels2=128),
        #one image served by a deep network: some eighty short launches in a row
        dict(name='resnet50_1_call', program='resnet50', way='call', batch=1, size=224),
        #the headline: a batch of images, arguments resident
        dict(name='resnet50_64', program='resnet50', way='replay', batch=64, size=224),
        #the same served: images from the host, logits and labels back
        dict(name='resnet50_64_call', program='resnet50', way='call', batch=64, size=224),
        #a training step of the deep network, forward, backward and update
        dict(name='resnet50_train_64', program='resnet50_train', way='replay', batch=64, size=224),
        #a large draw of random numbers
        dict(name='rng_uniform_16m', program='rng_uniform', way='replay', rows=4096, cols=4096),
        #embedding rows looked up, and their gradients added back into a table
        dict(name='gather_scatter_256k', program='gather_scatter', way='replay', rows=65536, cols=256, lookups=8192, bag=32),
        #class scores to probabilities and labels, rows of no round length
        dict(name='softmax_labels_1000', program='softmax_labels', way='replay', rows=65536, cols=1000),
    ]


def _log_int(rng, low, high):
    return min(high, max(low, int(round(low * (high / low) ** rng.random()))))


def _width(rng, low, high):
    '''A number of features: mostly a multiple of 8, at times any number.'''
    n = _log_int(rng, low, high)
    return n if rng.random() < 0.3 else max(8, n // 8 * 8)


def draw(rng):
    program = rng.choice(('affine', 'mlp', 'mlp_train', 'conv_block', 'convnet_train', 'resnet50', 'resnet50', 'resnet50_train',
                          'rng_uniform', 'gather_scatter', 'softmax_labels', 'normalised_residual'))
    way = 'replay'
    case = dict(program=program)
    if program == 'affine':
        way = 'call'
        case.update(batch=_log_int(rng, 1, 256), features=_width(rng, 16, 1024), outputs=_width(rng, 8, 512))
    elif program in ('mlp', 'mlp_train'):
        way = rng.choice(('call', 'replay')) if program == 'mlp' else 'replay'
        case.update(batch=_log_int(rng, 16, 8192), features=_width(rng, 64, 2048), hidden=_width(rng, 64, 2048),
                    hidden2=_width(rng, 32, 1024), classes=_log_int(rng, 2, 200))
    elif program == 'conv_block':
        size, channels = _log_int(rng, 7, 112), _width(rng, 16, 512)
        most = int(16e6 // (size * size * channels)) + 1
        case.update(batch=_log_int(rng, 1, max(2, min(256, most))), size=size, channels=channels)
    elif program == 'convnet_train':
        case.update(batch=_log_int(rng, 8, 128), size=_log_int(rng, 24, 128), channels=_width(rng, 16, 96), channels2=_width(rng, 32, 192))
    elif program in ('resnet50', 'resnet50_train'):
        size = rng.choice((rng.randint(96, 224), 224))
        way = rng.choice(('call', 'replay')) if program == 'resnet50' else 'replay'
        case.update(batch=_log_int(rng, 1 if program == 'resnet50' else 4, 64), size=size)
    elif program == 'rng_uniform':
        case.update(rows=_log_int(rng, 64, 4096), cols=_log_int(rng, 63, 8191))
    elif program == 'gather_scatter':
        case.update(rows=_log_int(rng, 1000, 131072), cols=_width(rng, 16, 512), lookups=_log_int(rng, 128, 8192), bag=rng.randint(1, 32))
    elif program == 'softmax_labels':
        cols = _log_int(rng, 10, 4096)
        case.update(rows=_log_int(rng, 64, max(65, min(65536, (1 << 26) // cols))), cols=cols)
    else:
        size, channels = _log_int(rng, 7, 112), _width(rng, 16, 512)
        most = int(5e7 // (size * size * channels)) + 1
        case.update(batch=_log_int(rng, 1, max(2, min(256, most))), size=size, channels=channels)
    case['way'] = way
    return case


# ------------------------------------------------------------------ a pass

class _InHBM:
    '''A result array of a recorded program where it lies in HBM (bool and unsigned words as int32).'''
    def __init__(self, buffer):
        kind = '<f4' if buffer.dtype == np.float32 else '<i4'
        self.owner = buffer
        self.__cuda_array_interface__ = dict(shape=buffer.shape, typestr=kind, data=(buffer.tensor.device_ptr(), False), version=2)


def _frozen(leaf):
    if isinstance(leaf, np.ndarray):
        leaf.flags.writeable = False
    return leaf


def prepare(case, seed):
    f, inputs = _program(case), _inputs(case, seed)
    if case['way'] == 'call':
        #the weights a server holds do not change: read-only arrays. (The affine layer's come with every call.)
        if case['program'] != 'affine':
            inputs[0] = tree_util.tree_map(_frozen, inputs[0])
        return dict(call=vkjax_amd.wrap(f, frontend='minijax'), inputs=inputs)
    program = JaxprInterpreter(mj.make_jaxpr(f)(*inputs))
    program.upload_inputs(*inputs)
    #a kernel is looked for in one code object after the other; the status of the last one that does not hold it would be
    #reported by torch's next call in its own name
    ctypes.CDLL('libamdhip64.so.7').hipGetLastError()
    outputs = [torch.as_tensor(_InHBM(b), device='cuda') for b in program.output_buffers]
    return dict(program=program, outputs=outputs)


def run(state):
    if 'call' in state:
        return state['call'](*state['inputs'])
    state['program'].replay(1)
    return state['outputs']


# ------------------------------------------------------------------ what a pass cannot do without

def _conv_layers(size):
    '''(output positions of one image, kernel elements) of every convolution of ResNet-50, and the size of its last features.'''
    half = lambda n: -(-n // 2)
    s = half(size)
    layers = [(s * s, 7 * 7 * 3 * 64)]
    s, cin = half(s), 64
    for blocks, width, stride in W.RESNET50_STAGES:
        for b in range(blocks):
            t = half(s) if b == 0 and stride == 2 else s
            layers += [(s * s, cin * width), (t * t, 9 * width * width), (t * t, width * 4 * width)]
            if b == 0:
                layers.append((t * t, cin * width * 4))
            s, cin = t, width * 4
    return layers, s, cin


def work(case):
    p = case['program']
    if p == 'affine':
        m, k, n = case['batch'], case['features'], case['outputs']
        return dict(bytes=4 * (m * k + k * n + n + m * n), flops=2 * m * k * n)
    if p in ('mlp', 'mlp_train'):
        m, sizes = case['batch'], (case['features'], case['hidden'], case['hidden2'], case['classes'])
        macs = sum(a * b for a, b in zip(sizes, sizes[1:]))
        weights = macs + sum(sizes[1:])
        if p == 'mlp':
            return dict(bytes=4 * (m * sizes[0] + weights + m * sizes[-1] + m), flops=2 * m * macs)
        return dict(bytes=4 * (m * (sizes[0] + sizes[-1]) + 2 * weights), flops=2 * m * (3 * macs - sizes[0] * sizes[1]))
    if p == 'conv_block':
        n, s, c = case['batch'], case['size'], case['channels']
        pooled = -(-s // 2)
        return dict(bytes=4 * (n * s * s * c + 9 * c * c + 4 * c + n * pooled * pooled * c), flops=2 * n * s * s * 9 * c * c)
    if p == 'convnet_train':
        n, s, c1, c2 = case['batch'], case['size'], case['channels'], case['channels2']
        s1 = (s - 1) // 2 + 1                                        #strided convolution, padding 1
        s2 = (s1 - 2) // 2 + 1                                       #3x3 pooling, one row of padding behind
        first, second = n * s1 * s1 * 27 * c1, n * s2 * s2 * 9 * c1 * c2
        weights = 27 * c1 + 9 * c1 * c2 + 2 * c1 + 10 * c2 + 10
        return dict(bytes=4 * (n * s * s * 3 + 10 * n + 2 * weights), flops=2 * (2 * first + 3 * second))
    if p in ('resnet50', 'resnet50_train'):
        n, (layers, _, last) = case['batch'], _conv_layers(case['size'])
        macs = sum(positions * kernel for positions, kernel in layers) + last * 1000
        weights = sum(kernel for _, kernel in layers) + last * 1000 + 1000
        image = case['size'] ** 2 * 3
        if p == 'resnet50':
            return dict(bytes=4 * (n * image + weights + n * 1001), flops=2 * n * macs)
        stem = layers[0][0] * layers[0][1]
        return dict(bytes=4 * (n * (image + 1000) + 2 * weights), flops=2 * n * (3 * macs - stem))
    if p == 'rng_uniform':
        return dict(bytes=4 * case['rows'] * case['cols'], flops=0)
    if p == 'gather_scatter':
        n, rows, cols = case['lookups'] * case['bag'], case['rows'], case['cols']
        #the rows that are looked up are read and written, the updates read, the table of sums written
        return dict(bytes=4 * (3 * n * cols + n + rows * cols), flops=n * cols)
    if p == 'softmax_labels':
        return dict(bytes=4 * (2 * case['rows'] * case['cols'] + case['rows']), flops=5 * case['rows'] * case['cols'])
    n = case['batch'] * case['size'] ** 2 * case['channels']
    return dict(bytes=4 * (3 * n + case['batch'] * case['channels']), flops=5 * n)


def tolerance(case):
    #What 32-bit sums in another order give: the 2-norm of the difference to the same path in 64 bits over the 2-norm of the
    #result, measured at the listed and some drawn sizes (of the worst output), times about four. The updated weights of the
    #deep network are the loosest: they are mostly gradient, and a gradient that passes fifty layers changes by up to 1.4e-3
    #when sums are rounded in another way (ReLU and pooling choose differently where values all but tie).
    p = case['program']
    if p == 'rng_uniform':
        return 'exact'
    return {'affine': dict(rel=1e-6), 'mlp': dict(rel=1e-6), 'mlp_train': dict(rel=1e-6), 'conv_block': dict(rel=1e-6),
            'convnet_train': dict(rel=1e-6), 'resnet50': dict(rel=2e-6), 'resnet50_train': dict(rel=6e-3), 'gather_scatter': dict(rel=2e-7),
            'softmax_labels': dict(rel=4e-7, differ=1e-4), 'normalised_residual': dict(rel=3e-7)}[p]
