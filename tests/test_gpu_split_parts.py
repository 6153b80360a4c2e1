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


def scaled(shape, factor):
    return (rng.standard_normal(shape) * factor).astype(np.float32)


#x, w by their factors: numbers whose parts a bf16 cannot hold (below 2^-102 = 2e-31), down to those with few bits themselves
SMALL = [(1e-32, 1e30), (1e-36, 1e30), (1e-38, 1e20), (1e-42, 1e25), (1e30, 1e-36), (1e25, 1e-42), (1e-36, 1.0), (1e-20, 1e-17), (1e-19, 1e-19)]


def assert_fp32_error(y, x, w):
    '''At most two roundings per product of two k and one per 64 k, parts left out and cut sums below that: (K + K / 64 + 17) 2^-24 sum |x||w|;
    numbers too small for 24 bits of their own are off by half of 2^-149 per rounding.'''
    K_    = x.shape[1]
    exact = x.astype(np.float64) @ w.astype(np.float64)
    limit = (np.abs(x).astype(np.float64) @ np.abs(w).astype(np.float64)) * (K_ + K_ / 64 + 17) * 2.0 ** -24 + (K_ + 1) * 2.0 ** -150
    assert (np.abs(y - exact) <= limit).all(), np.max(np.abs(y - exact) / limit)
    return np.linalg.norm(y - exact)


@pytest.mark.gpu
@pytest.mark.parametrize('fx,fw', SMALL)
def test_small_operands_keep_their_bits(fx, fw):
    '''Some rows (columns) of small numbers, some of zeros, some of ordinary ones; in the 2-norm no further off than fp32 products are.'''
    K_, M, N = 320, 200, 72
    x, w = scaled((M, K_), fx), scaled((K_, N), fw)
    x[5], x[130:140], w[:, 3], w[:, 40:44] = 0, 0, 0, 0
    x[7], x[150] = scaled((2, K_), 1.0)
    x[9, :200], x[160, 1:] = 0, 0
    dot = lambda x, w: jnp.dot(x, w)
    wg  = lambda x, g: mj.lax.dot_general(x, g, (((0,), (0,)), ((), ())))
    def result(f, a, b, **choice):
        with K.overrides(**choice):
            return vkjax_amd.wrap(f, frontend='minijax')(a, b)
    fp32 = assert_fp32_error(result(dot, x, w, conv_split=False), x, w)
    for tile in K.CONV_SPLIT_TILES:
        for slices in (1, 3):
            print(f'case: {fx} {fw}, tile {tile}, {slices} slices', flush=True)
            assert assert_fp32_error(result(dot, x, w, conv_split=tile, conv_split_slices=slices), x, w) <= 1.05 * fp32
    xt   = np.ascontiguousarray(x.T)
    fp32 = assert_fp32_error(result(wg, xt, w, wgrad_split=False), x, w)
    for tile in K.WGRAD_SPLIT_TILES:
        for slices in (1, 3):
            print(f'case: kernel gradient, {fx} {fw}, tile {tile}, {slices} slices', flush=True)
            assert assert_fp32_error(result(wg, xt, w, wgrad_split=tile, wgrad_slices=slices), x, w) <= 1.05 * fp32


@pytest.mark.gpu
@pytest.mark.parametrize('tile', list(K.CONV_SPLIT_TILES))
@pytest.mark.parametrize('stride,dilation,padding', [((1, 1), (1, 1), 'SAME'), ((2, 2), (1, 1), 'SAME'), ((1, 1), (2, 3), 'VALID')])
def test_small_images(tile, stride, dilation, padding):
    '''Rows that are windows of an image, parts of them outside it: powers of two below 2^-102, so that every product is exact.'''
    f = lambda x, k: mj.lax.conv_general_dilated(x, k, stride, padding, rhs_dilation=dilation, dimension_numbers=('NHWC', 'HWIO', 'NHWC'))
    x = (rng.randint(-4, 5, size=(2, 15, 14, 32)) * 2.0 ** -145).astype(np.float32)
    x[1, 3:9] = 0
    k = (rng.randint(-3, 4, size=(3, 3, 32, 40)) * 2.0 ** 100).astype(np.float32)
    with K.overrides(conv_split=False):
        expected = vkjax_amd.wrap(f, frontend='minijax')(x, k)
    with K.overrides(conv_split=tile):
        assert np.array_equal(vkjax_amd.wrap(f, frontend='minijax')(x, k), expected) and (expected != 0).any()


@pytest.mark.gpu
@pytest.mark.parametrize('large', (2.0 ** 48, 2.0 ** 49, 2.0 ** 103, 2.0 ** 104, 2.0 ** 120, 3.4e38))
def test_large_kernel_operands(large):
    '''Weights around the largest that are packed in three parts, and beyond: integers times powers of two, so that every result is exact.'''
    x, w = rng.randint(-4, 5, size=(140, 160)).astype(np.float32), rng.randint(-3, 4, size=(160, 70)).astype(np.float32)
    w[77, 5], w[100, 69], w[100, 68] = large, -large, large
    x[:, 77], x[:, 100] = np.sign(x[:, 77]), np.sign(x[:, 100])
    results = []
    for choice in list(K.CONV_SPLIT_TILES) + [False]:
        with K.overrides(conv_split=choice):
            results.append(vkjax_amd.wrap(lambda x, w: jnp.dot(x, w), frontend='minijax')(x, w))
    exact = x.astype(np.float64) @ w.astype(np.float64)
    small = np.arange(70)[~np.isin(np.arange(70), (5, 68, 69))]
    for y in results:
        assert np.array_equal(y[:, small], exact[:, small])
        assert np.allclose(y, exact, rtol=160 * 2.0 ** -24, atol=0)           #one rounding per term


@pytest.mark.gpu
@pytest.mark.parametrize('k', (16, 40, 64, 200))
def test_last_bits_of_small_rows(k):
    '''Rows of numbers whose last bits no bf16 part holds unless it is scaled, against weights of 1, one of them 2^48: that column's sums are the one
    number times 2^48, all others together are below the half of the last bit.'''
    x = (2.0 ** -112 * (1 + (2 * rng.randint(0, 2 ** 22, size=(130, k)) + 1) * 2.0 ** -23)).astype(np.float32)
    for at in sorted({0, 1, k // 2, k - 1}):
        for n in (0, 31, 32, 70):
            w = np.ones((k, 71), np.float32)
            w[at, n] = 2.0 ** 48
            for tile in K.CONV_SPLIT_TILES:
                with K.overrides(conv_split=tile):
                    y = vkjax_amd.wrap(lambda x, w: jnp.dot(x, w), frontend='minijax')(x, w)
                assert np.array_equal(y[:, n], x[:, at] * np.float32(2.0 ** 48)), (tile, at, n)
                assert_fp32_error(y, x, w)
