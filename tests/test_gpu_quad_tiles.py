'''The kernels whose four waves share a 32 x 32 tile: contractions around whole k steps and whole vectors, tiles handed to the XCDs row by row and column by
column, windows whose taps change within and between k steps. Whole numbers, so every result is exact.'''
import numpy as np
import pytest

import vkjax_amd
from vkjax_amd import kernels as K, minijax as mj
from tests.common import check_against_oracle

lax, nn, jnp = mj.lax, mj.nn, mj.numpy
rng = np.random.RandomState(11)


def ints(lo, hi, *s):
    return rng.randint(lo, hi, size=s).astype(np.float32)


def layer(x, w, mean, scale, beta, rest):
    return nn.relu((jnp.dot(x, w) - mean) * scale + beta + rest)


def kernels_of(fn):
    return [l.kernel for l in list(fn._jaxpr_interpreters.values())[0].launches]


#one k step of 128 to six, each with the step before and behind full, and remainders within a vector and within a wave's slice of 32
LENGTHS = (1, 3, 4, 31, 32, 33, 96, 97, 127, 128, 129, 160, 255, 256, 257, 384, 386, 512, 515, 640, 641, 768)


@pytest.mark.gpu
@pytest.mark.parametrize('xcd', ('columns', 0, 'ranges'))
@pytest.mark.parametrize('m,n', ((2, 20), (33, 68), (65, 290), (200, 33)))
def test_contractions(m, n, xcd):
    for k in LENGTHS:
        print('four waves per tile:', m, k, n, xcd, flush=True)
        args = [ints(-4, 5, m, k), ints(-3, 4, k, n), ints(-5, 5, n), ints(1, 4, n), ints(-9, 9, n), ints(-50, 50, m, n)]
        with K.overrides(conv_ksplit=True, conv_k_splits=1, conv_xcd_columns=xcd, conv_dense_rows=False):
            _, _, fn = check_against_oracle(layer, args, exact=True)
        assert kernels_of(fn) == ['conv_gemm_32x32x128_ks4'], kernels_of(fn)


@pytest.mark.gpu
@pytest.mark.parametrize('xcd', ('columns', 0))
@pytest.mark.parametrize('shares', (2, 5))
def test_shared_tiles(shares, xcd):
    for m, k, n in ((33, 700, 100), (70, 1300, 260)):
        args = [ints(-4, 5, m, k), ints(-3, 4, k, n), ints(-5, 5, n), ints(1, 4, n), ints(-9, 9, n), ints(-50, 50, m, n)]
        with K.overrides(conv_ksplit=True, conv_shares=shares, conv_k_splits=1, conv_xcd_columns=xcd):
            _, _, fn = check_against_oracle(layer, args, exact=True)
        assert kernels_of(fn) == ['conv_gemm_32x32x128_ks4_shared'], kernels_of(fn)


#(input, kernel, strides, padding, dilation of the kernel): taps outside on each side, on none, windows wider than the image
WINDOWS = [((1, 7, 5, 128), (3, 3, 128, 40), (1, 1), 'SAME', (1, 1)), ((2, 9, 8, 128), (3, 2, 128, 33), (2, 1), 'SAME', (1, 1)), ((1, 9, 9, 256), (3, 3, 256, 36), (1, 2), 'VALID', (2, 3)),
           ((2, 6, 7, 64), (5, 5, 64, 32), (1, 1), 'SAME', (1, 1)), ((1, 4, 3, 192), (3, 5, 192, 20), (1, 1), ((3, 2), (0, 4)), (1, 1)), ((3, 5, 5, 128), (1, 1, 128, 64), (2, 2), 'VALID', (1, 1)),
           ((1, 6, 6, 128), (2, 3, 128, 32), (1, 1), ((1, 0), (2, 1)), (3, 1))]


@pytest.mark.gpu
@pytest.mark.parametrize('general', (False, True))
@pytest.mark.parametrize('x,w,strides,padding,dilation', WINDOWS)
def test_windows(x, w, strides, padding, dilation, general):
    print('four waves per tile:', x, w, strides, padding, dilation, general, flush=True)
    def f(x, w, shift):
        return nn.relu(lax.conv_general_dilated(x, w, strides, padding, rhs_dilation=dilation, dimension_numbers=('NHWC', 'HWIO', 'NHWC')) + shift)
    with K.overrides(conv_ksplit=True, conv_k_splits=1, conv_shares=1, conv_b_general=general, conv_split=False):
        _, _, fn = check_against_oracle(f, [ints(-4, 5, *x), ints(-3, 4, *w), ints(-9, 9, w[-1])], exact=True)
    if not (general and x[-1] % 128):
        assert '_ks4' in kernels_of(fn)[-1], kernels_of(fn)


def test_ranges_of_tiles():
    '''Column by column where that fetches less.'''
    choose = K.choose_conv_xcd_columns
    assert choose(256, 2048, 2048, 8, 64) == choose(196, 1024, 256, 7, 32) == choose(784, 128, 1152, 25, 4, 784 * 128) == K.CONV_XCD_COLUMNWISE
    assert choose(1000, 300, 784, 32, 10) == choose(600, 256, 1024, 19, 8) == 0


def transposed(x, w, mean, scale, beta, rest):
    return nn.relu((lax.dot_general(x, w, (((1,), (1,)), ((), ()))) - mean) * scale + beta + rest)


@pytest.mark.gpu
@pytest.mark.parametrize('shares', (1, 3))
@pytest.mark.parametrize('m,n', ((2, 20), (65, 291), (300, 36)))
def test_transposed_kernel_operand(m, n, shares):
    for k in LENGTHS:
        print('four waves per tile, transposed:', m, k, n, shares, flush=True)
        args = [ints(-4, 5, m, k), ints(-3, 4, n, k), ints(-5, 5, n), ints(1, 4, n), ints(-9, 9, n), ints(-50, 50, m, n)]
        with K.overrides(conv_ksplit=True, conv_k_splits=1, conv_shares=shares, conv_dense_rows=False, conv_split=False):
            _, _, fn = check_against_oracle(transposed, args, exact=True)
        names = kernels_of(fn)
        assert names == ['conv_gemm_32x32x128_ks4t' + ('_shared' if shares > 1 and k > 128 else '')] or (k == 1 and len(names) == 1), names


@pytest.mark.gpu
def test_what_lies_behind_a_row_is_not_added():
    '''A contraction that ends within a vector: the next row's first value, infinite here, stays out of both operands.'''
    x, w = ints(-4, 5, 40, 131), ints(-3, 4, 36, 131)
    x[1:, 0] = w[1::2, 0] = np.inf
    x[0, 0], w[0, 0] = 1, 1
    def f(x, w): return lax.dot_general(x, w, (((1,), (1,)), ((), ())))
    with K.overrides(conv_ksplit=True, conv_k_splits=1, conv_dense_rows=False, conv_split=False):
        fn  = vkjax_amd.wrap(f, frontend='minijax')
        got = fn(x, w)
    assert kernels_of(fn) == ['conv_gemm_32x32x128_ks4t_shared'] or kernels_of(fn) == ['conv_gemm_32x32x128_ks4t'], kernels_of(fn)
    assert np.array_equal(got[0, 0::2], w[0::2] @ x[0])


def clipped(x, w):
    return jnp.minimum(lax.dot_general(x, w, (((1,), (1,)), ((), ()))), np.float32(6)) / np.float32(2)


@pytest.mark.parametrize('k,launches', ((1000, 2), (512, 2), (200, 1)))
def test_long_products_stay_with_four_waves(k, launches):
    '''A chain that these kernels have no epilogue for stays a launch of its own behind a long product.'''
    interp, _ = vkjax_amd.wrap(clipped, frontend='minijax', plan_only=True)._get_or_create_jaxpr_interpreter([ints(-4, 5, 64, k), ints(-3, 4, 2048, k)])
    names = [l.kernel for l in interp.launches]
    assert len(names) == launches and ('_ks4t' in names[0]) == (launches == 2), names


@pytest.mark.gpu
@pytest.mark.parametrize('k', (200, 1000))
def test_long_products_with_another_chain(k):
    check_against_oracle(clipped, [ints(-4, 5, 64, k), ints(-3, 4, 2048, k)], exact=True)


def swapped(x, w):
    return lax.conv_general_dilated(x, w, (1, 1), 'SAME', dimension_numbers=('NHWC', 'HWOI', 'NHWC'))


@pytest.mark.parametrize('features,copied', ((32, False), (64, True), (256, True)))
def test_long_products_of_few_rows_read_a_copy(features, copied):
    '''A kernel operand with its last two dimensions swapped is copied into the dense layout where the contraction is long, however few the rows are.'''
    interp, _ = vkjax_amd.wrap(swapped, frontend='minijax', plan_only=True)._get_or_create_jaxpr_interpreter([ints(-4, 5, 1, 5, 6, features), ints(-3, 4, 3, 3, 64, features)])
    assert any('transpose' in l.kernel or l.kernel.startswith('ew_') for l in interp.launches[:1]) == copied, [l.kernel for l in interp.launches]


@pytest.mark.gpu
@pytest.mark.parametrize('features', (32, 64, 256))
def test_swapped_kernel_operands(features):
    check_against_oracle(swapped, [ints(-4, 5, 1, 5, 6, features), ints(-3, 4, 3, 3, 64, features)], exact=True)


#classes of an input dilated by 2 (or 3): every second (third) row and column of the result, each from its own taps
CLASSES = [((2, 5, 6, 256), (3, 3, 256, 36), ((1, 2), (2, 1)), 2), ((1, 4, 9, 512), (2, 3, 512, 64), ((2, 1), (1, 1)), 2), ((3, 3, 3, 1024), (1, 1, 1024, 68), ((0, 1), (0, 1)), 2),
           ((1, 3, 4, 128), (5, 5, 128, 32), ((4, 3), (2, 4)), 3), ((8, 5, 5, 512), (3, 3, 512, 512), ((1, 2), (1, 2)), 2)]


@pytest.mark.gpu
@pytest.mark.parametrize('x,w,padding,dilation', CLASSES)
def test_classes_of_a_dilated_input(x, w, padding, dilation):
    print('dilated input:', x, w, padding, dilation, flush=True)
    def f(x, w):
        return lax.conv_general_dilated(x, w, (1, 1), padding, lhs_dilation=(dilation, dilation), dimension_numbers=('NHWC', 'HWIO', 'NHWC'))
    _, _, fn = check_against_oracle(f, [ints(-4, 5, *x), ints(-3, 4, *w)], exact=True)
    assert 'conv_gemm_32x32x128_ks4_strided' in kernels_of(fn), kernels_of(fn)
