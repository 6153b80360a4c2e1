'''Average pooling and its gradient with the steps around them in one launch (pool2d_sum): the bits of the separate launches over
windows, strides, borders and channels at which taps fall outside or between the elements.'''
import numpy as np
import pytest

import vkjax_amd
from vkjax_amd import minijax as mj
from vkjax_amd.minijax import lax

jnp = mj.numpy
f32 = np.float32


def pooled(x, window, strides, padding):
    return lax.reduce_window(x, 0.0, lax.add, (1,) + window + (1,), (1,) + strides + (1,), padding)


def kernels_of(f, args, **kwargs):
    interp, _ = vkjax_amd.wrap(f, frontend='minijax', **kwargs)._get_or_create_jaxpr_interpreter(args)
    return [l.kernel for l in interp.launches]


#(batch, y, x, channels, window, strides, padding)
SHAPES = [(1, 2, 2, 4, (2, 2), (2, 2), 'VALID'), (3, 5, 7, 8, (2, 2), (2, 2), 'VALID'), (2, 6, 5, 12, (2, 2), (1, 1), 'SAME'), (2, 9, 8, 64, (3, 3), (2, 2), 'SAME'),
          (1, 7, 7, 132, (3, 3), (3, 3), 'VALID'), (2, 3, 3, 4, (3, 3), (1, 1), 'SAME'), (5, 11, 4, 20, (2, 2), (3, 3), 'VALID'), (1, 24, 24, 128, (2, 2), (2, 2), 'VALID')]


def mean_pool(x, c, window, strides, padding):
    return pooled(x, window, strides, padding) / f32(window[0] * window[1]), c * pooled(x * c, window, strides, padding)


def relu_mean_pool_gradient(x, target, window, strides, padding):
    loss = lambda x, target: jnp.sum(pooled(mj.nn.relu(x), window, strides, padding) / f32(window[0] * window[1]) * target)
    return mj.grad(loss)(x, target)


def global_mean_gradient(x, scores, window, strides, padding):
    '''One value per image and channel behind the pooling: its gradient is the same for all positions.'''
    loss = lambda x, scores: jnp.sum(jnp.mean(pooled(mj.nn.relu(x), window, strides, padding) / f32(7), axis=(1, 2)) * scores)
    return mj.grad(loss)(x, scores)


def case(shape, seed=0):
    B, H, W_, C, window, strides, padding = shape
    rng = np.random.default_rng(seed)
    x   = rng.standard_normal((B, H, W_, C)).astype(f32)
    bound = lambda f: (lambda *args: f(*args, window, strides, padding))
    ny, nx = (((n - k) // s + 1) if padding == 'VALID' else -(-n // s) for n, k, s in zip((H, W_), window, strides))
    return [(bound(mean_pool), (x, f32(0.3))), (bound(relu_mean_pool_gradient), (x, rng.standard_normal((B, ny, nx, C)).astype(f32))),
            (bound(global_mean_gradient), (x, rng.standard_normal((B, C)).astype(f32)))]


def test_launches():
    (means, args), (gradient, gargs), (spread, sargs) = case(SHAPES[-1])
    kernels = kernels_of(means, args, plan_only=True)
    assert kernels == ['pool2d_sum_2x2_v4'] * 2, kernels
    for f, a in ((gradient, gargs), (spread, sargs)):
        kernels = kernels_of(f, a, plan_only=True)
        assert kernels.count('pad_nd_pool2d_sum_2x2_v4') == 1 and not any(k.startswith('pad_nd_v') for k in kernels), kernels
    #other values between the elements, an array in between that something else reads, a whole array behind the sum: not taken over
    x, one = args[0], f32(1)
    spread_by = lambda v: (lambda x: pooled(lax.pad(x, v, ((0, 0, 0), (1, 1, 1), (1, 1, 1), (0, 0, 0))), (2, 2), (1, 1), 'VALID'))
    assert any(k.startswith('pad_nd_v') for k in kernels_of(spread_by(one), (x,), plan_only=True))
    assert not any(k.startswith('pad_nd_v') for k in kernels_of(spread_by(f32(0)), (x,), plan_only=True))
    for f in (lambda x: (lambda h: (h, pooled(h, (2, 2), (2, 2), 'VALID')))(x / f32(3)), lambda x: (lambda s: s * s)(pooled(x, (2, 2), (1, 1), 'SAME')),
              lambda x: pooled(x / x, (2, 2), (2, 2), 'VALID'), lambda x: (lambda p: p / p)(pooled(x, (2, 2), (2, 2), 'VALID'))):
        assert not any('pool2d_sum' in k for k in kernels_of(f, (x,), plan_only=True))


@pytest.mark.gpu
@pytest.mark.parametrize('shape', SHAPES, ids=str)
def test_every_bit(shape):
    for k, (f, args) in enumerate(case(shape)):
        for special in (False, True):
            print('window sum', shape, k, special, flush=True)
            if special:
                args = tuple(np.array(a) for a in args)
                for a in args:
                    flat = a.reshape(-1)
                    flat[0] = -0.0
                    if flat.size > 8:
                        flat[1], flat[5], flat[-1] = np.inf, np.nan, -np.inf
            got, expected = (mj.tree_util.tree_leaves(vkjax_amd.wrap(f, frontend='minijax', fuse=fuse)(*args)) for fuse in (True, False))
            for a, b in zip(got, expected):
                number = ~np.isnan(b)
                assert np.array_equal(a, b, equal_nan=True) and np.array_equal(np.signbit(a)[number], np.signbit(b)[number]), (shape, k)
