'''What is left of a number when its nearest bf16 has been taken off (csrc/kernels/split_bf16.h) has to be exact: operands of which all
three parts matter, over many exponents, leave the products' error at that of 64-bit sums rounded once.'''
import numpy as np
import pytest

import vkjax_amd
from vkjax_amd import kernels as K
from vkjax_amd import minijax as mj

jnp = mj.numpy
rng = np.random.RandomState(31)


@pytest.mark.gpu
@pytest.mark.parametrize('low,high', ((-100, -40), (-20, 20), (40, 120)))
def test_single_products_keep_all_24_bits(low, high):
    '''Each row of x holds one number beside zeros and the kernel operand is a permutation scaled by powers of two: every result is one
    operand times 2^n, to the last bit. Neighbours of a number, which share its instruction, hold numbers of other sizes.'''
    x = np.ldexp(rng.uniform(1, 2, size=(256, 64)), rng.randint(low, high, size=(256, 64))).astype(np.float32) * rng.choice([-1, 1], size=(256, 64)).astype(np.float32)
    w = np.zeros((64, 64), np.float32)
    w[rng.permutation(64), np.arange(64)] = np.ldexp(1.0, rng.randint(-3, 4, size=64))
    expected = (x.astype(np.float64) @ w.astype(np.float64)).astype(np.float32)
    for tile in K.CONV_SPLIT_TILES:
        with K.overrides(conv_split=tile):
            assert np.array_equal(vkjax_amd.wrap(lambda x, w: jnp.dot(x, w), frontend='minijax')(x, w), expected), tile
    for tile in K.WGRAD_SPLIT_TILES:
        with K.overrides(wgrad_split=tile):
            xt = np.ascontiguousarray(np.concatenate([x.T, np.zeros((64, 256), np.float32)]))             #contracted over 128 rows
            wt = np.concatenate([w, np.zeros((64, 64), np.float32)])
            y  = vkjax_amd.wrap(lambda x, g: mj.lax.dot_general(x, g, (((0,), (0,)), ((), ()))), frontend='minijax')(xt, wt)
            assert np.array_equal(y, expected), tile
