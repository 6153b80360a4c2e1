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


def few_terms(rows, K, n):
    x = np.zeros((rows, K), np.float32)
    for i in range(rows):
        x[i, rng.permutation(K)[:n]] = rng.standard_normal(n)
    return x


@pytest.mark.gpu
@pytest.mark.parametrize('n', (1, 2, 3, 16))
def test_sums_of_few_terms_are_cut_off_once_per_product_behind_the_first(n):
    '''The matrix cores cut a sum off below its last bit (an error under 2^-23 of it). The small partial products of a k step are added before
    the large one, so a sum's first term meets the cut once at full size (the two adds before it, at 2^-8 of it at most), and every later one
    six times: 2^-23 (6 (n - 1) + 1 + 2 2^-8). The partial products left out are below 2 2^-9 2^-17 = 2^-25 of a term (a part is at
    most 2^-9 of what the one before stands for, the third 2^-17), and each of at most n sums of k tiles is rounded once into the accumulator
    (2^-24; the first of them has nothing to be rounded with). All in units of sum |x||w|.'''
    x, w  = few_terms(256, 256, n), rng.standard_normal((256, 96)).astype(np.float32)
    exact = x.astype(np.float64) @ w.astype(np.float64)
    limit = (np.abs(x).astype(np.float64) @ np.abs(w).astype(np.float64)) * \
            ((6 * (n - 1) + 1 + 2.0 ** -7) * 2.0 ** -23 + 2.0 ** -25 + (n - 1) * 2.0 ** -24)
    for tile in K.CONV_SPLIT_TILES:
        with K.overrides(conv_split=tile):
            y = vkjax_amd.wrap(lambda x, w: jnp.dot(x, w), frontend='minijax')(x, w)
        assert (np.abs(y - exact) <= limit).all(), (tile, np.max(np.abs(y - exact) / np.maximum(limit, 1e-300)))
    for tile in K.WGRAD_SPLIT_TILES:
        with K.overrides(wgrad_split=tile):
            y = vkjax_amd.wrap(lambda x, g: mj.lax.dot_general(x, g, (((0,), (0,)), ((), ()))), frontend='minijax')(np.ascontiguousarray(x.T), w)
        assert (np.abs(y - exact) <= limit).all(), (tile, np.max(np.abs(y - exact) / np.maximum(limit, 1e-300)))


@pytest.mark.gpu
@pytest.mark.parametrize('value', (np.inf, np.nan, 3.4e38))
def test_finite_sums_keep_their_bits_beside_others(value):
    '''Data whose sums are rounded: an operand that is not finite (or beyond the largest bf16) in one row changes that row only.'''
    x, w  = rng.standard_normal((200, 160)).astype(np.float32), rng.standard_normal((160, 96)).astype(np.float32)
    other = x.copy()
    other[37, 21] = value
    rest  = np.arange(200) != 37
    for tile in K.CONV_SPLIT_TILES:
        for slices in (1, 2):
            with K.overrides(conv_split=tile, conv_split_slices=slices):
                fn = vkjax_amd.wrap(lambda x, w: jnp.dot(x, w), frontend='minijax')
                before, after = fn(x, w), fn(other, w)
            assert np.array_equal(before[rest], after[rest]) and not np.array_equal(before[37], after[37]), (tile, slices)
    for tile in K.WGRAD_SPLIT_TILES:
        with K.overrides(wgrad_split=tile):
            fn = vkjax_amd.wrap(lambda x, g: mj.lax.dot_general(x, g, (((0,), (0,)), ((), ()))), frontend='minijax')
            before, after = fn(np.ascontiguousarray(x.T), w), fn(np.ascontiguousarray(other.T), w)
        assert np.array_equal(before[rest], after[rest]) and not np.array_equal(before[37], after[37]), tile
