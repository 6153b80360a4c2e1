'''Row programs (rows.hip) over the row lengths at which their variants begin and end and numbers of rows that leave a wave
or a block partly empty: the bits of the separate launches, and 64-bit values within fp32's reach.'''
import numpy as np
import pytest

import vkjax_amd
from vkjax_amd import minijax as mj, workloads as W
from vkjax_amd.minijax import lax

pytestmark = pytest.mark.gpu
jnp = mj.numpy

#a row of one value per lane holds 64, of one vector per lane 256 values: both sides of each end, and what lies between
LENGTHS = [2, 3, 4, 7, 8, 10, 31, 32, 33, 63, 64, 65, 100, 127, 252, 255, 256, 257, 260, 511, 1000, 1001, 1020, 1023, 1024]


def loss_and_gradient(x, onehot):
    return mj.value_and_grad(W.softmax_cross_entropy)(x, onehot)


def normalised(x, scale, shift, weight):
    '''Rows to mean 0 and variance 1, then a scale and a shift per column: vectors over both dimensions, several results.'''
    mean = jnp.sum(x, axis=1, keepdims=True) / np.float32(x.shape[1])
    d    = x - mean
    var  = jnp.sum(d * d, axis=1, keepdims=True) / np.float32(x.shape[1])
    y    = d * lax.rsqrt(var + np.float32(1e-5)) * scale + shift
    return y * weight, mean, jnp.max(y, axis=1), jnp.sum(lax.tanh(y) * weight, axis=1)


def run(f, args, name):
    fused, unfused = (vkjax_amd.wrap(f, frontend='minijax', fuse=fuse) for fuse in (True, False))
    got, expected  = fused(*args), unfused(*args)
    kernels = [l.kernel for l in list(fused._jaxpr_interpreters.values())[0].launches]
    assert sum(k.startswith('rows_v') for k in kernels) == 1 and len(kernels) <= name[1], (name, kernels)
    for a, b in zip(mj.tree_util.tree_leaves(got), mj.tree_util.tree_leaves(expected)):
        assert np.array_equal(a, b, equal_nan=True), (name, a, b)
    return got


@pytest.mark.parametrize('cols', LENGTHS)
def test_loss_and_gradient(cols):
    rng = np.random.default_rng(cols)
    for rows in (2, 67):
        print(f'cross-entropy {rows} x {cols}', flush=True)
        x = (rng.standard_normal((rows, cols)) * 3).astype(np.float32)
        onehot = np.eye(cols, dtype=np.float32)[rng.integers(0, cols, rows)]
        loss, grad = run(loss_and_gradient, [x, onehot], ('cross-entropy', 5))
        x64 = x.astype(np.float64)
        p   = np.exp(x64 - x64.max(axis=1, keepdims=True))
        p  /= p.sum(axis=1, keepdims=True)
        #x - max is rounded to fp32 (2^-24 of at most 30) before exp, the sum of a row a few times: below 1e-5 of a probability
        assert np.allclose(grad, (p - onehot) / rows, rtol=1e-5, atol=1e-6 / rows)
        assert np.isclose(loss, -np.mean(np.log((p * onehot).sum(axis=1))), rtol=1e-5)
        #infinities, NaN, zeros of both signs, the lowest number
        x[0, cols - 1], x[1, 0] = np.nan, np.inf
        if rows > 2:
            x[2, :], x[3, cols // 2], x[4, :], x[5, :], x[6, 0] = -np.inf, -np.inf, -0.0, np.where(np.arange(cols) % 2, 0.0, -0.0), -3.4e38
        run(loss_and_gradient, [x, onehot], ('cross-entropy', 5))


@pytest.mark.parametrize('cols', [2, 5, 64, 65, 256, 300, 768, 1022, 1024])
@pytest.mark.parametrize('rows', [3, 250])
def test_vectors_over_both_dimensions(cols, rows):
    rng  = np.random.default_rng(cols * rows)
    args = [rng.standard_normal(s).astype(np.float32) for s in ((rows, cols), (cols,), (cols,), (rows, 1))]
    run(normalised, args, ('normalised', 2))


def test_rows_of_a_stack():
    '''Rows of more dimensions than two, one operand of which is read through a transposition.'''
    rng = np.random.default_rng(3)
    def f(x, t):
        e = lax.exp(x - jnp.max(x, axis=2, keepdims=True))
        s = jnp.sum(e, axis=2, keepdims=True)
        return lax.log(s) * np.float32(2), jnp.sum(e * lax.transpose(t, (2, 0, 1)), axis=2)
    args = [rng.standard_normal((6, 7, 20)).astype(np.float32), rng.standard_normal((7, 20, 6)).astype(np.float32)]
    fused, unfused = (vkjax_amd.wrap(f, frontend='minijax', fuse=fuse)(*args) for fuse in (True, False))
    for a, b in zip(fused, unfused):
        assert np.array_equal(a, b)
