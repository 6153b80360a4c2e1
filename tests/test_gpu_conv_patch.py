'''The kernels for 3 x 3 windows that hold a patch of the input in LDS (conv_patch_sums in csrc/kernels/conv_split.h): integer-valued
data make every product and sum exact; on random data they are no further from 64-bit sums than the kernels that load every tap anew.'''
import numpy as np
import pytest

import vkjax_amd
from vkjax_amd import kernels as K, minijax as mj
from vkjax_amd.jaxpr_interpreter import JaxprInterpreter

from .common import check_against_oracle

lax, nn, jnp = mj.lax, mj.nn, mj.numpy
rng = np.random.RandomState(29)
conv = lambda x, k: lax.conv_general_dilated(x, k, (1, 1), 'SAME', dimension_numbers=('NHWC', 'HWIO', 'NHWC'))


def ints(shape, low=-4, high=5):
    return rng.randint(low, high, size=shape).astype(np.float32)


def kernels_of(fn):
    return [l.kernel for l in list(fn._jaxpr_interpreters.values())[0].launches if l.kernel.startswith('conv_gemm')]


#[batch, H, W, features], columns: images narrower, as wide and wider than a tile's rows reach, the widest there is room for, one row or one
#column of pixels, tiles that end inside an image, between two and in the first rows of the next, features of one to several turns of the loop
SHAPES = [([1, 1, 1, 32], 1), ([3, 5, 1, 32], 40), ([2, 1, 9, 64], 64), ([1, 2, 64 - 1, 32], 33), ([2, 7, 7, 96], 129), ([5, 14, 14, 64], 70), ([1, 28, 28, 32], 128),
          ([2, 5, 56, 64], 64), ([2, 9, 63, 32], 65), ([4, 3, 43, 160], 5), ([9, 2, 2, 64], 31), ([1, 128, 1, 32], 32), ([1, 129, 2, 64], 64)]


@pytest.mark.gpu
@pytest.mark.parametrize('tile', list(K.CONV_SPLIT_TILES))
@pytest.mark.parametrize('xs,columns', SHAPES, ids=[f'{"x".join(map(str, s))} {n}' for s, n in SHAPES])
def test_image_and_tile_edges(tile, xs, columns):
    x, k = ints(xs), ints([3, 3, xs[3], columns], -3, 4)
    for slices in (1, 2, 3):
        if slices > xs[3] // 32:
            continue
        print(f'case: {xs} {columns}, tile {tile}, {slices} slices', flush=True)
        with K.overrides(conv_split=tile, conv_split_slices=slices, conv_patch=True):
            _, _, fn = check_against_oracle(conv, [x, k], exact=True)
        assert kernels_of(fn) == [f'conv_gemm_split_{tile}_patch']
        first = fn(x, k)                                      #the slices' counters are zeros again
        assert np.array_equal(first, fn(x, k))


@pytest.mark.gpu
@pytest.mark.parametrize('tile', list(K.CONV_SPLIT_TILES))
def test_epilogues_and_reversed_kernels(tile):
    x, k, r, v = ints([2, 14, 13, 64]), ints([3, 3, 64, 72], -3, 4), ints([2, 14, 13, 72], -50, 50), 2.0 ** ints([72], -2, 3)
    bn      = lambda x, k, r, v: nn.relu((conv(x, k) - v) * v + v + r)
    two     = lambda x, k, r, v: (lambda c: (nn.relu(c * v), c))(conv(x, k) - v)
    steps   = lambda x, k, r, v: (((conv(x, k) + v) * v - r) * 0.5 + r) * v
    turned  = lambda x, k, r, v: conv(r, lax.rev(lax.transpose(k, (0, 1, 3, 2)), (0, 1))) + x
    for f in (bn, two, steps):
        for slices in (1, 2):
            with K.overrides(conv_split=tile, conv_split_slices=slices, conv_patch=True):
                _, _, fn = check_against_oracle(f, [x, k, r, v], exact=True)
            assert len(kernels_of(fn)) == 1 and '_patch' in kernels_of(fn)[0], kernels_of(fn)
    r, k = ints([2, 14, 13, 96]), ints([3, 3, 64, 96], -3, 4)
    with K.overrides(conv_split=tile, conv_patch=True):
        _, _, fn = check_against_oracle(turned, [x, k, r, v], exact=True)
    assert kernels_of(fn) == [f'conv_gemm_split_{tile}_patch']


@pytest.mark.gpu
@pytest.mark.parametrize('tile', list(K.CONV_SPLIT_TILES))
def test_values_that_are_not_finite_stay_where_they_are(tile):
    '''An infinity, a NaN and a number beyond the parts' range reach the results whose windows they lie in, and no other: those next to them, in
    the row before and behind and in the next image stay what they are.'''
    x, k = ints([3, 9, 20, 64]), ints([3, 3, 64, 70], -3, 4)
    x[0, 0, 0, 3], x[0, 8, 19, 40], x[1, 4, 0, 63], x[2, 8, 7, 0] = np.inf, np.nan, -np.inf, 1e37
    k[1, 1, 5, 69] = np.inf
    with K.overrides(conv_split=False):
        expected = vkjax_amd.wrap(conv, frontend='minijax')(x, k)
    for slices in (1, 2):
        with K.overrides(conv_split=tile, conv_split_slices=slices, conv_patch=True):
            y = vkjax_amd.wrap(conv, frontend='minijax')(x, k)
        same = np.isfinite(expected)
        assert np.array_equal(np.isfinite(y), same)
        #3e38 times a small weight: finite sums beyond 2^80 are computed with fp32 products, whose order of terms is another
        assert np.allclose(y[same], expected[same], rtol=576 * 2.0 ** -24, atol=0)
        assert np.array_equal(y[~same], expected[~same], equal_nan=True)


def error(y, x, k):
    '''The 2-norm of the difference to 64-bit sums over that of the result.'''
    xp = np.pad(x.astype(np.float64), ((0, 0), (1, 1), (1, 1), (0, 0)))
    exact = sum(xp[:, r:r + x.shape[1], s:s + x.shape[2]] @ k[r, s].astype(np.float64) for r in range(3) for s in range(3))
    return np.linalg.norm(y - exact) / np.linalg.norm(exact)


@pytest.mark.gpu
@pytest.mark.parametrize('features', (32, 64, 256, 512))
@pytest.mark.parametrize('kind', ('normal', 'activations', 'small', 'sparse', 'all positive'))
def test_error_against_64_bits(features, kind):
    '''No larger than with every tap loaded anew; for sums of which every term is positive, no larger than that of fp32 products (three steps are summed
    before they are added up, not four: where sums only grow, the additions are what is rounded, and there are 4/3 as many).'''
    x, k = (rng.standard_normal(s).astype(np.float32) for s in ((4, 28, 28, features), (3, 3, features, 64)))
    if kind in ('activations', 'all positive'):
        x = np.abs(x)
    if kind == 'all positive':
        k = np.abs(k)
    elif kind == 'small':
        x, k = x * np.float32(1e-36), k * np.float32(1e30)
    elif kind == 'sparse':
        x = (x * (rng.rand(*x.shape) < 1 / 16)).astype(np.float32)
    def of(**choice):
        with K.overrides(**choice):
            return error(vkjax_amd.wrap(conv, frontend='minijax')(x, k), x, k)
    for tile in K.CONV_SPLIT_TILES:
        here, there = of(conv_split=tile, conv_patch=True), of(conv_split=False) if kind == 'all positive' else of(conv_split=tile, conv_patch=False)
        print(f'{kind}, {features} features, {tile}: {here:.3g}, {there:.3g}', flush=True)
        assert here <= 1.02 * there                            #(norms over 200704 results: they scatter by 0.5 %)


def test_where_the_patch_kernels_apply():
    '''Plan only.'''
    def launches(x, k, f=conv, **choice):
        with K.overrides(**choice):
            return [l.kernel for l in JaxprInterpreter(mj.make_jaxpr(f)(np.zeros(x, np.float32), np.zeros(k, np.float32)), plan_only=True).launches if l.kernel.startswith('conv_gemm')]
    patch = lambda *a, **c: ['_patch' in k for k in launches(*a, **c)] == [True]
    assert patch((64, 28, 28, 128), (3, 3, 128, 128)) and patch((16, 56, 56, 64), (3, 3, 64, 64)) and patch((64, 7, 7, 512), (3, 3, 512, 512))
    assert patch((16, 63, 63, 64), (3, 3, 64, 64)) and not patch((16, 64, 64, 64), (3, 3, 64, 64))                   #256 positions
    assert not patch((64, 28, 28, 144), (3, 3, 144, 128)) and not patch((64, 28, 28, 128), (5, 5, 128, 128))          #features, window
    strided = lambda x, k: lax.conv_general_dilated(x, k, (2, 2), 'SAME', dimension_numbers=('NHWC', 'HWIO', 'NHWC'))
    valid   = lambda x, k: lax.conv_general_dilated(x, k, (1, 1), 'VALID', dimension_numbers=('NHWC', 'HWIO', 'NHWC'))
    dilated = lambda x, k: lax.conv_general_dilated(x, k, (1, 1), 'SAME', rhs_dilation=(2, 2), dimension_numbers=('NHWC', 'HWIO', 'NHWC'))
    assert not any(patch((64, 28, 28, 128), (3, 3, 128, 128), f) for f in (strided, valid, dilated))
    assert not patch((64, 28, 28, 128), (3, 3, 128, 128), conv_split='128x64') and not patch((64, 28, 28, 128), (3, 3, 128, 128), conv_patch=False)
