'''Steps of gradient descent stored by the column sum that computes the gradient, and weight gradients computed in the layout of
the weights: the bits of the separate launches where they add in one order, 64-bit values within fp32's reach.'''
import numpy as np
import pytest

import vkjax_amd
from vkjax_amd import minijax as mj
from vkjax_amd.minijax import lax

jnp = mj.numpy
RATE = np.float32(0.03)


def kernels_of(f, args, **kwargs):
    wrapped = vkjax_amd.wrap(f, frontend='minijax', **kwargs)
    interp, _ = wrapped._get_or_create_jaxpr_interpreter(args)
    return [l.kernel for l in interp.launches]


def sums_step(params, arrays):
    '''One update by a column sum per parameter, with the rate on either side.'''
    return [p - RATE * jnp.sum(a, axis=0) if k % 2 else p - jnp.sum(a, axis=0) * RATE for k, (p, a) in enumerate(zip(params, arrays))]


def sums_args(shapes, seed=0):
    rng = np.random.default_rng(seed)
    return ([rng.standard_normal(c).astype(np.float32) for _, c in shapes], [rng.standard_normal(s).astype(np.float32) for s in shapes])


#one row and one step of 4 thread rows more or less, one vector and one lane's width more or less, split and unsplit sums
SHAPES = [(2, 2), (2, 3), (3, 4), (4, 5), (5, 8), (16, 10), (17, 64), (63, 100), (64, 256), (65, 257), (127, 260), (1000, 10), (1000, 300), (1536, 64), (1537, 64), (5000, 1000)]


def test_updates_are_planned():
    for shape in SHAPES:
        kernels = kernels_of(sums_step, sums_args([shape]), plan_only=True)
        assert kernels[-1].startswith('reduce_cols_fsum_update_v') and not any(k.startswith('ew_chain') for k in kernels), (shape, kernels)
    kernels = kernels_of(sums_step, sums_args([(7, 64), (20, 100), (9, 7), (30, 10), (63, 1000)]), plan_only=True)
    assert kernels == ['reduce_cols_fsum_batch_update'], kernels
    #a gradient that is returned or read again, other signs, a rate per column and a sum over the leading of three dimensions' rows
    kept = [lambda p, a: (lambda g: (p - RATE * g, g))(jnp.sum(a, axis=0)), lambda p, a: (lambda g: (p - RATE * g) * g)(jnp.sum(a, axis=0)),
            lambda p, a: RATE * jnp.sum(a, axis=0) - p, lambda p, a: p + RATE * jnp.sum(a, axis=0), lambda p, a: p - p * jnp.sum(a, axis=0)]
    p, a = np.ones(12, np.float32), np.ones((9, 12), np.float32)
    for f in kept:
        assert not any('update' in k for k in kernels_of(f, (p, a), plan_only=True))


@pytest.mark.gpu
@pytest.mark.parametrize('shapes', [[s] for s in SHAPES] + [SHAPES, SHAPES[::2]], ids=lambda s: '+'.join(f'{r}x{c}' for r, c in s[:2]))
def test_updates_keep_every_bit(shapes):
    print('updates', shapes, flush=True)
    params, arrays = sums_args(shapes, seed=len(shapes))
    got      = vkjax_amd.wrap(sums_step, frontend='minijax')(params, arrays)
    expected = vkjax_amd.wrap(sums_step, frontend='minijax', fuse=False)(params, arrays)
    for p, a, g, e in zip(params, arrays, got, expected):
        assert np.array_equal(g, e)
        #a sum of n terms in fp32 is off by at most n roundings of the sum of their magnitudes, the step by two more
        a64 = a.astype(np.float64)
        bound = 2.0**-24 * (len(a) * float(RATE) * np.abs(a64).sum(axis=0) + 3 * (np.abs(p) + float(RATE) * np.abs(a64.sum(axis=0))))
        assert np.all(np.abs(g - (p - float(RATE) * a64.sum(axis=0))) <= bound)
    params[0][0], arrays[0][0, -1], arrays[-1][0, 0] = np.inf, np.nan, -np.inf
    got      = vkjax_amd.wrap(sums_step, frontend='minijax')(params, arrays)
    expected = vkjax_amd.wrap(sums_step, frontend='minijax', fuse=False)(params, arrays)
    for g, e in zip(got, expected):
        assert np.array_equal(g, e, equal_nan=True)


def weight_gradient(w, x, cot):
    return lax.transpose(lax.dot_general(cot, x, (((0,), (0,)), ((), ()))), (1, 0))


def weight_step(w, x, cot):
    return w - RATE * weight_gradient(w, x, cot)


#(rows, inputs, outputs): both sides of the 128 rows from which the rows are cut into ranges, tile edges, ragged sizes
PRODUCTS = [(1, 3, 5), (5, 64, 10), (127, 10, 100), (128, 10, 100), (129, 65, 63), (200, 1, 7), (200, 7, 1), (1000, 100, 10), (513, 129, 257), (4096, 64, 128)]


def test_weight_gradients_are_computed_in_the_layout_of_the_weights():
    for rows, n_in, n_out in PRODUCTS:
        args = [np.ones(s, np.float32) for s in ((n_in, n_out), (rows, n_in), (rows, n_out))]
        for f in (weight_gradient, weight_step):
            fused, unfused = (kernels_of(f, args, plan_only=True, fuse=fuse) for fuse in (True, False))
            assert len(fused) < len(unfused) and not any('transpose' in k for k in fused), (rows, n_in, n_out, fused)
    #a product that is read in its own layout as well keeps it
    both = lambda w, x, cot: (lambda g: (g, lax.transpose(g, (1, 0))))(lax.dot_general(cot, x, (((0,), (0,)), ((), ()))))
    assert [o.shape for o in mj.tree_util.tree_leaves(vkjax_amd.wrap(both, frontend='minijax', plan_only=True)._get_or_create_jaxpr_interpreter(args)[0].output_buffers)] == [(128, 64), (64, 128)]


@pytest.mark.gpu
@pytest.mark.parametrize('rows,n_in,n_out', PRODUCTS)
def test_weight_gradients(rows, n_in, n_out):
    print('weight gradient', rows, n_in, n_out, flush=True)
    rng = np.random.default_rng(rows)
    w, x, cot = (rng.standard_normal(s).astype(np.float32) for s in ((n_in, n_out), (rows, n_in), (rows, n_out)))
    exact = x.astype(np.float64).T @ cot
    #a product of n terms in fp32 is off by at most n roundings of the sum of their magnitudes
    bound = (rows + 2) * 2.0**-24 * (np.abs(x).astype(np.float64).T @ np.abs(cot))
    for fuse in (True, False):
        got = vkjax_amd.wrap(weight_gradient, frontend='minijax', fuse=fuse)(w, x, cot)
        assert got.shape == (n_in, n_out) and np.all(np.abs(got - exact) <= bound), fuse
        new = vkjax_amd.wrap(weight_step, frontend='minijax', fuse=fuse)(w, x, cot)
        assert np.all(np.abs(new - (w - float(RATE) * exact)) <= float(RATE) * bound + 3 * 2.0**-24 * (np.abs(w) + float(RATE) * np.abs(exact))), fuse


def relu_backward(pre, g):
    '''The gradient through a ReLU and of the bias in front of it, with the gradient read again.'''
    m = jnp.where(pre > np.float32(0.25), g, np.float32(0))
    return m, jnp.sum(m, axis=0)


#unsplit sums end at 1536 rows; blocks of 256 columns, of 8 vectors or values, and what lies beside them
RELU_SHAPES = [(2, 2), (3, 4), (17, 10), (63, 64), (64, 65), (127, 100), (127, 256), (128, 256), (129, 257), (1000, 300), (1000, 7), (1536, 40), (1537, 40), (4099, 8), (700, 1028)]


def test_relu_backward_with_its_sum_is_planned():
    for shape in RELU_SHAPES:
        x = np.ones(shape, np.float32)
        kernels = kernels_of(relu_backward, (x, x), plan_only=True)
        assert kernels[0].startswith('relu_backward_v') and len(kernels) == (2 if shape[0] > 1536 else 1), (shape, kernels)
    #values of the mask per column, or sums along the other dimension: the launches stay apart
    other = [lambda x, g: (lambda m: (m, jnp.sum(m, axis=0)))(jnp.where(x > x[0], g, np.float32(0))),
             lambda x, g: (lambda m: (m, jnp.sum(m, axis=1)))(jnp.where(x > np.float32(0), g, np.float32(0)))]
    for f in other:
        assert not any(k.startswith('relu_backward') for k in kernels_of(f, (np.ones((9, 12), np.float32),) * 2, plan_only=True))


@pytest.mark.gpu
@pytest.mark.parametrize('shape', RELU_SHAPES, ids=str)
def test_relu_backward_keeps_every_bit(shape):
    print('relu backward', shape, flush=True)
    rng  = np.random.default_rng(shape[0])
    x, g = (rng.standard_normal(shape).astype(np.float32) for _ in range(2))
    x[0, 0], g[1, 1], x[1, 0], g[0, 1] = np.nan, np.inf, np.float32(0.25), -0.0
    got, expected = (vkjax_amd.wrap(relu_backward, frontend='minijax', fuse=fuse)(x, g) for fuse in (True, False))
    for a, b in zip(got, expected):
        assert np.array_equal(a, b, equal_nan=True)
    assert np.array_equal(got[0], np.where(x > np.float32(0.25), g, np.float32(0)), equal_nan=True)


def scaled_sums(x, c):
    '''A change of sign behind a mean: of rows, of columns, of everything, with values known before and with one that is not.'''
    n = np.float32(x.shape[0])
    return [-(jnp.sum(x, axis=1) / c), -(jnp.sum(x, axis=0) / n), -(jnp.sum(x) / np.float32(x.size)), jnp.sum(x, axis=0) / c, c * jnp.sum(x)]


@pytest.mark.gpu
@pytest.mark.parametrize('shape', [(2, 3), (5, 64), (127, 12), (128, 10), (1000, 10), (3, 8192), (4, 40000), (5000, 33)], ids=str)
def test_scaled_sums_keep_every_bit(shape):
    x, c = np.random.default_rng(1).standard_normal(shape).astype(np.float32), np.float32(7)
    x[0, 0], x[1, 1] = 0, -0.0
    got, expected = (vkjax_amd.wrap(scaled_sums, frontend='minijax', fuse=fuse)(x, c) for fuse in (True, False))
    kernels = kernels_of(scaled_sums, (x, c), plan_only=True)
    assert shape[0] > 1536 or x.size > 4096 or not any(k.startswith('ew_chain') for k in kernels), kernels       #(split sums keep theirs)
    for a, b in zip(got, expected):
        assert np.array_equal(a, b)


def known_scalars(x):
    '''Values that are known before anything runs, and one that is not: quotients that need rounding, signed zeros, an overflow and
    an underflow (which the device computes).'''
    neg, div, mul = lax.neg, lax.div, lax.mul
    f = np.float32
    values = [div(neg(f(1)), f(1000)), div(f(1), f(3)), mul(div(f(2), f(3)), f(0.1)), neg(f(0)), div(neg(f(0)), f(5)), mul(f(3e38), f(10)), div(f(1e-38), f(10))]
    return [x * v for v in values] + [values[0]]


def test_known_scalars_cost_no_launch():
    kernels = kernels_of(lambda x: x * lax.div(lax.neg(np.float32(1)), np.float32(1000)), (np.ones(64, np.float32),), plan_only=True)
    assert len(kernels) == 1, kernels


@pytest.mark.gpu
def test_known_scalars_keep_every_bit():
    x = np.linspace(-3, 3, 65).astype(np.float32)
    got, expected = (vkjax_amd.wrap(known_scalars, frontend='minijax', fuse=fuse)(x) for fuse in (True, False))
    for a, b in zip(got, expected):
        assert np.array_equal(np.asarray(a, np.float32).view(np.uint32), np.asarray(b, np.float32).view(np.uint32))
