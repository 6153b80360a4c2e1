'''3 x 3 windows over a number of features that is no multiple of 32, on the bf16 matrix cores.'''
import numpy as np
import pytest

import vkjax_amd
from vkjax_amd import kernels as K, minijax as mj
from vkjax_amd.jaxpr_interpreter import JaxprInterpreter

lax, nn, jnp = mj.lax, mj.nn, mj.numpy
rng = np.random.RandomState(77)
RAGGED = 'conv_gemm_split_128x64_ragged'


def conv(x, k):
    return lax.conv_general_dilated(x, k, (1, 1), 'SAME', dimension_numbers=('NHWC', 'HWIO', 'NHWC'))


def residual(x, k, mean, scale, beta, rest):
    return nn.relu((conv(x, k) - mean) * scale + beta + rest)


def clipped(x, k, mean):
    return jnp.minimum(nn.relu(conv(x, k) - mean), np.float32(6))


def kernels_of(fn):
    return [l.kernel for l in list(fn._jaxpr_interpreters.values())[0].launches if l.kernel.startswith('conv_gemm')]


def exact_sums(x, k):
    xp = np.pad(x.astype(np.float64), ((0, 0), (1, 1), (1, 1), (0, 0)))
    return sum(xp[:, r:r + x.shape[1], s:s + x.shape[2]] @ k[r, s].astype(np.float64) for r in range(3) for s in range(3))


#one to three words behind whole vectors, one to seven vectors behind groups of 32 and 16; ragged rows and columns, images of one row and column, the widest patch, slices
SHAPES = [((1, 3, 5, 4), 3), ((2, 9, 7, 17), 40), ((1, 11, 11, 105), 105), ((3, 1, 33, 33), 70), ((3, 33, 1, 47), 64), ((1, 63, 63, 20), 9), ((2, 10, 12, 52), 130), ((4, 7, 7, 200), 33), ((1, 8, 8, 447), 65)]


@pytest.mark.gpu
@pytest.mark.parametrize('xs,columns', SHAPES, ids=lambda v: 'x'.join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_integers_are_exact(xs, columns):
    print('ragged features:', xs, columns, flush=True)
    ints = lambda lo, hi, *s: rng.randint(lo, hi, size=s).astype(np.float32)
    x, k, mean, scale, beta = ints(-8, 9, *xs), ints(-6, 7, 3, 3, xs[3], columns), ints(-5, 5, columns), ints(1, 4, columns), ints(-9, 9, columns)
    rest  = ints(-50, 50, *xs[:3], columns)
    sums  = exact_sums(x, k)
    wants = [(conv, [x, k], sums), (residual, [x, k, mean, scale, beta, rest], np.maximum((sums - mean) * scale + beta + rest, 0)),
             (clipped, [x, k, mean], np.minimum(np.maximum(sums - mean, 0), 6))]
    with K.overrides(conv_ragged=True):
        for f, args, want in wants:
            fn = vkjax_amd.wrap(f, frontend='minijax')
            for _ in range(2):
                assert np.array_equal(fn(*args), want.astype(np.float32))
            assert kernels_of(fn)[0].startswith(RAGGED), kernels_of(fn)


@pytest.mark.gpu
@pytest.mark.parametrize('features', (21, 44, 105))
def test_what_lies_behind_the_last_feature_is_not_seen(features):
    '''Sums beside a value that is not finite keep their bits, those that see it are what fp32 products give; numbers near both ends of the range.'''
    print('ragged, not finite:', features, flush=True)
    x, k = rng.standard_normal((2, 9, 8, features)).astype(np.float32), rng.standard_normal((3, 3, features, 40)).astype(np.float32)
    with K.overrides(conv_ragged=True):
        fn = vkjax_amd.wrap(conv, frontend='minijax')
        y  = fn(x, k)
        assert kernels_of(fn) == [RAGGED]
        for odd in (np.inf, -np.inf, np.nan, np.float32(3e38), np.float32(1e-44)):
            z = x.copy()
            z[0, 4, 3, 0] = odd                                   #a position's first feature lies behind the one before it
            got, seen = fn(z, k), np.zeros(y.shape, bool)
            seen[0, 3:6, 2:5] = True
            assert np.array_equal(got[~seen], y[~seen])
            with np.errstate(all='ignore'):
                want = exact_sums(z, k).astype(np.float32)
            finite = np.isfinite(want)
            assert np.array_equal(np.isfinite(got), finite) and np.array_equal(got[~finite], want[~finite], equal_nan=True)
            assert np.allclose(got[finite], want[finite], rtol=1e-4, atol=1e-4)


@pytest.mark.gpu
@pytest.mark.parametrize('kind', (0.004, 1 / 16, 1 / 4, 'normal', 'small', 'all positive', 'one weight'))
@pytest.mark.parametrize('xs,columns', [((4, 28, 28, 72), 64), ((3, 14, 14, 250), 96), ((1, 7, 7, 477), 480), ((8, 24, 24, 25), 64)], ids=lambda v: 'x'.join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_error_against_64_bits(xs, columns, kind):
    '''No larger than that of the fp32 kernels; a number: the share of the input that is not zero.'''
    x, k = rng.standard_normal(xs).astype(np.float32), rng.standard_normal((3, 3, xs[3], columns)).astype(np.float32)
    if isinstance(kind, float):
        x *= rng.random_sample(x.shape) < kind
    elif kind == 'small':
        x, k = x * np.float32(1e-36), k * np.float32(1e30)
    elif kind == 'all positive':
        x, k = np.abs(x), np.abs(k)
    elif kind == 'one weight':
        k *= (np.argsort(rng.random_sample((9 * xs[3], columns)), axis=0) < 1).reshape(k.shape)
    exact = exact_sums(x, k)
    def error(**choice):
        with K.overrides(**choice):
            fn = vkjax_amd.wrap(conv, frontend='minijax')
            y  = fn(x, k)
        assert (kernels_of(fn) == [RAGGED]) == ('conv_ragged' in choice)
        return np.linalg.norm(y - exact) / np.linalg.norm(exact)
    here, there = error(conv_ragged=True), error(conv_split=False)
    print(f'{xs} {columns}, {kind}: {here:.4g}, {there:.4g}', flush=True)
    assert here <= 1.01 * there


@pytest.mark.parametrize('xs,columns,taken', [((1, 8, 8, 22), 22, 1), ((4, 14, 14, 17), 17, 0), ((1, 8, 8, 104), 104, 1), ((60, 28, 28, 100), 17, 0), ((4, 14, 14, 60), 60, 1), ((30, 14, 14, 72), 72, 0),
                                              ((60, 40, 40, 36), 36, 1), ((10, 40, 40, 60), 60, 0), ((4, 64, 64, 105), 105, 0), ((4, 14, 14, 64), 64, 0)])
def test_where_it_is_taken(xs, columns, taken):
    zeros  = lambda *s: np.broadcast_to(np.float32(0), s)
    interp = JaxprInterpreter(mj.make_jaxpr(conv)(zeros(*xs), zeros(3, 3, xs[3], columns)), plan_only=True)
    assert (RAGGED in [l.kernel for l in interp.launches]) == bool(taken)


@pytest.mark.parametrize('images,size,features,columns,layout,there', [
    (11, 31, 397, 397, 'HWIO', True), (1, 8, 104, 104, 'HWIO', True), (64, 7, 200, 200, 'HWIO', True), (60, 40, 60, 60, 'HWIO', True), (47, 23, 44, 216, 'HWIO', True), (60, 40, 22, 22, 'HWIO', True),
    (15, 38, 52, 78, 'HWOI', True), (113, 22, 8, 288, 'HWIO', False), (17, 54, 36, 88, 'HWIO', False), (78, 11, 40, 224, 'HWIO', False), (36, 15, 68, 360, 'HWIO', False),
    (38, 35, 100, 32, 'HWIO', False), (27, 26, 104, 24, 'HWIO', False), (38, 56, 8, 218, 'HWIO', False), (93, 58, 72, 4, 'HWIO', False), (107, 43, 52, 24, 'HWIO', False), (24, 14, 33, 152, 'HWIO', False), (79, 18, 68, 68, 'HWIO', True), (98, 26, 36, 36, 'HWIO', False), (15, 38, 40, 144, 'HWOI', True), (125, 43, 80, 8, 'HWOI', False), (7, 31, 120, 120, 'HWIO', True), (10, 18, 104, 264, 'HWIO', False), (125, 32, 4, 286, 'HWOI', False)])
def test_where_they_pay(images, size, features, columns, layout, there):
    '''Plan only: not where so many features are padding, or columns, that the fp32 kernels are ahead.'''
    def f(x, w):
        return lax.conv_general_dilated(x, w, (1, 1), ((1, 1), (1, 1)), dimension_numbers=('NHWC', layout, 'NHWC'))
    zeros   = lambda *s: np.broadcast_to(np.float32(0), s)
    kernel  = zeros(3, 3, columns, features) if layout == 'HWOI' else zeros(3, 3, features, columns)
    program = JaxprInterpreter(mj.make_jaxpr(f)(zeros(images, size, size, features), kernel), plan_only=True)
    assert (RAGGED in [l.kernel for l in program.launches]) == there, [l.kernel for l in program.launches]
