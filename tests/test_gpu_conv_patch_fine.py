'''The kernel for 3 x 3 windows that holds a patch of the input in LDS and keeps two sums (FINE in csrc/kernels/conv_split.h), which serves
products that were fp32 ones: integer-valued data make every product and sum exact; on other data, however many of a sum's terms are zero,
its results are as close to 64-bit sums as those of the fp32 kernels.'''
import numpy as np
import pytest

import vkjax_amd
from vkjax_amd import kernels as K, minijax as mj
from vkjax_amd.jaxpr_interpreter import JaxprInterpreter

from .common import check_against_oracle
from .test_gpu_conv_patch import SHAPES, conv, ints, kernels_of

lax, nn, jnp = mj.lax, mj.nn, mj.numpy
rng = np.random.RandomState(37)
FINE = 'conv_gemm_split_128x64_patch_fine'


@pytest.mark.gpu
@pytest.mark.parametrize('xs,columns', SHAPES, ids=[f'{"x".join(map(str, s))} {n}' for s, n in SHAPES])
def test_image_and_tile_edges(xs, columns):
    x, k = ints(xs), ints([3, 3, xs[3], columns], -3, 4)
    for slices in (1, 2, 3):
        if slices > xs[3] // 32:
            continue
        print(f'case: {xs} {columns}, {slices} slices', flush=True)
        with K.overrides(conv_split_slices=slices, conv_patch='fine'):
            _, _, fn = check_against_oracle(conv, [x, k], exact=True)
        assert kernels_of(fn) == [FINE]
        first = fn(x, k)                                      #the slices' counters are zeros again
        assert np.array_equal(first, fn(x, k))


@pytest.mark.gpu
def test_epilogues():
    x, k, r, v = ints([2, 14, 13, 64]), ints([3, 3, 64, 72], -3, 4), ints([2, 14, 13, 72], -50, 50), 2.0 ** ints([72], -2, 3)
    bn     = lambda x, k, r, v: nn.relu((conv(x, k) - v) * v + v + r)
    steps  = lambda x, k, r, v: (((conv(x, k) + v) * v - r) * 0.5 + r) * v
    masked = lambda x, k, r, v: jnp.where(r > 0.0, conv(x, k), 0.0) * v
    for f, name in ((bn, FINE), (steps, FINE + '_steps'), (masked, FINE)):
        for slices in (1, 2):
            with K.overrides(conv_split_slices=slices, conv_patch='fine'):
                _, _, fn = check_against_oracle(f, [x, k, r, v], exact=True)
            assert kernels_of(fn) == [name]


@pytest.mark.gpu
def test_values_that_are_not_finite_stay_where_they_are():
    x, k = ints([3, 9, 20, 64]), ints([3, 3, 64, 70], -3, 4)
    x[0, 0, 0, 3], x[0, 8, 19, 40], x[1, 4, 0, 63], x[2, 8, 7, 0] = np.inf, np.nan, -np.inf, 1e37
    k[1, 1, 5, 69] = np.inf
    with K.overrides(conv_split=False):
        expected = vkjax_amd.wrap(conv, frontend='minijax')(x, k)
    for slices in (1, 2):
        with K.overrides(conv_split_slices=slices, conv_patch='fine'):
            y = vkjax_amd.wrap(conv, frontend='minijax')(x, k)
        same = np.isfinite(expected)
        #3e38 times a small weight: finite sums beyond 2^80 are computed with fp32 products, whose order of terms is another
        assert np.array_equal(np.isfinite(y), same) and np.allclose(y[same], expected[same], rtol=576 * 2.0 ** -24, atol=0)
        assert np.array_equal(y[~same], expected[~same], equal_nan=True)


@pytest.mark.gpu
@pytest.mark.parametrize('kind', (0.001, 0.004, 0.016, 1 / 16, 1 / 8, 1 / 4, 1 / 2, 'normal', 'small', 'all positive', 'one weight'))
@pytest.mark.parametrize('xs,columns', [([4, 28, 28, 64], 64), ([3, 14, 14, 256], 96), ([1, 7, 7, 480], 480), ([8, 7, 7, 512], 512), ([8, 24, 24, 32], 64)],
                         ids=lambda v: 'x'.join(map(str, v)) if isinstance(v, list) else str(v))
def test_error_against_64_bits(xs, columns, kind):
    '''No larger than that of the fp32 kernels, with the slices that the plan chooses; a number: the share of the input that is not zero.'''
    x, k = rng.standard_normal(xs).astype(np.float32), rng.standard_normal((3, 3, xs[3], columns)).astype(np.float32)
    if isinstance(kind, float):
        x *= rng.random_sample(x.shape) < kind
    elif kind == 'small':
        x, k = x * np.float32(1e-36), k * np.float32(1e30)
    elif kind == 'all positive':
        x, k = np.abs(x), np.abs(k)
    elif kind == 'one weight':
        k *= (np.argsort(rng.random_sample((9 * xs[3], columns)), axis=0) < 1).reshape(k.shape)
    xp = np.pad(x.astype(np.float64), ((0, 0), (1, 1), (1, 1), (0, 0)))
    exact = sum(xp[:, r:r + xs[1], s:s + xs[2]] @ k[r, s].astype(np.float64) for r in range(3) for s in range(3))
    def error(**choice):
        with K.overrides(**choice):
            fn = vkjax_amd.wrap(conv, frontend='minijax')
            y  = fn(x, k)
        assert (kernels_of(fn) == [FINE]) == ('conv_patch' in choice)
        return np.linalg.norm(y - exact) / np.linalg.norm(exact)
    here, there = error(conv_patch='fine'), error(conv_split=False)
    print(f'{xs} {columns}, {kind}: {here:.4g}, {there:.4g}', flush=True)
    assert here <= 1.01 * there


@pytest.mark.parametrize('xs,columns,kernel', [([16, 7, 7, 512], 512, FINE), ([15, 7, 7, 512], 512, None), ([64, 56, 56, 64], 32, FINE), ([1, 7, 7, 480], 480, FINE),
                                               ([1, 10, 10, 160], 40, FINE), ([2, 40, 40, 96], 64, FINE), ([9, 20, 20, 96], 96, None), ([8, 14, 14, 256], 256, None),
                                               ([1, 28, 28, 32], 128, None), ([64, 28, 28, 128], 128, 'conv_gemm_split_128x128_patch')])
def test_where_it_is_taken(xs, columns, kernel):
    '''Plan only: both sides of every line. What the bf16 kernels served before stays with the ones of one sum.'''
    zeros = lambda *s: np.broadcast_to(np.float32(0), s)
    interp = JaxprInterpreter(mj.make_jaxpr(conv)(zeros(*xs), zeros(3, 3, xs[3], columns)), plan_only=True)
    names  = [l.kernel for l in interp.launches if l.kernel.startswith('conv_gemm')]
    assert names == [kernel] if kernel else '_split' not in names[0], names


def test_pinned_to_the_patch_kernels():
    '''Plan only: wherever they apply, and nowhere else.'''
    zeros = lambda *s: np.broadcast_to(np.float32(0), s)
    pointwise = lambda x, k: lax.conv_general_dilated(x, k, (1, 1), 'VALID', dimension_numbers=('NHWC', 'HWIO', 'NHWC'))
    for choice, kernel in ((True, '_patch'), ('fine', '_patch_fine')):
        with K.overrides(conv_patch=choice):
            for f, window, expected in ((conv, 3, kernel), (pointwise, 1, None)):
                interp = JaxprInterpreter(mj.make_jaxpr(f)(zeros(2, 14, 14, 64), zeros(window, window, 64, 64)), plan_only=True)
                name,  = [l.kernel for l in interp.launches if l.kernel.startswith('conv_gemm')]
                assert name.endswith(expected) if expected else '_split' not in name, name


@pytest.mark.gpu
@pytest.mark.parametrize('share', (0.004, 1 / 16, 1.0))
@pytest.mark.parametrize('xs,columns', [([4, 7, 7, 1024], 256), ([12, 7, 7, 768], 512)], ids=lambda v: 'x'.join(map(str, v)) if isinstance(v, list) else str(v))
def test_error_beside_shared_tiles(xs, columns, share):
    '''Nor larger than that of the kernels whose blocks share a tile, which add shorter sums than one block does, and which would compute these products.'''
    x, k = rng.standard_normal(xs).astype(np.float32), rng.standard_normal((3, 3, xs[3], columns)).astype(np.float32)
    x   *= rng.random_sample(x.shape) < share
    xp   = np.pad(x.astype(np.float64), ((0, 0), (1, 1), (1, 1), (0, 0)))
    exact = sum(xp[:, r:r + xs[1], s:s + xs[2]] @ k[r, s].astype(np.float64) for r in range(3) for s in range(3))
    def error(kernel, **choice):
        with K.overrides(**choice):
            fn = vkjax_amd.wrap(conv, frontend='minijax')
            y  = fn(x, k)
        assert kernels_of(fn) == [kernel]
        return np.linalg.norm(y - exact) / np.linalg.norm(exact)
    here, there = error(FINE, conv_patch='fine'), error('conv_gemm_32x32x128_ks4_shared', conv_patch=False, conv_ragged=False)
    print(f'{xs} {columns}, {share}: {here:.4g}, {there:.4g}', flush=True)
    assert here <= 1.01 * there
