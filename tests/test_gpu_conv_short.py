'''The kernels for dense rows of at most 64 features (conv_short_body in csrc/kernels/conv_split.h): integer-valued data make every product and
sum exact, and on any data, however many of a sum's terms are zero, they are as close to 64-bit sums as the fp32 kernels.'''
import numpy as np
import pytest

import vkjax_amd
from vkjax_amd import kernels as K, minijax as mj
from vkjax_amd.jaxpr_interpreter import JaxprInterpreter

from .common import check_against_oracle

nn, jnp = mj.nn, mj.numpy
rng = np.random.RandomState(31)


def ints(shape, low=-4, high=5):
    return rng.randint(low, high, size=shape).astype(np.float32)


def kernels_of(fn):
    return [l.kernel for l in list(fn._jaxpr_interpreters.values())[0].launches if l.kernel.startswith('conv_gemm')]


#rows around one tile, a wave's second tile (256 blocks of 12 waves: from 98304 on) and none; features that fill a vector, a k tile, not all of
#two; columns around a block of 32, of 256, and groups of blocks that are not equally wide
SHAPES = [(33, 4, 17), (31, 64, 256), (32, 36, 32), (65, 60, 257), (1000, 64, 300), (98400, 32, 33), (40, 44, 1100), (8200, 64, 8200)]


@pytest.mark.gpu
@pytest.mark.parametrize('m,k,n', SHAPES)
def test_tile_edges(m, k, n):
    x, w = ints((m, k)), ints((k, n), -3, 4)
    with K.overrides(conv_short=True):
        fn = vkjax_amd.wrap(jnp.dot, frontend='minijax')
        y  = np.asarray(fn(x, w))
    assert kernels_of(fn) == ['conv_gemm_split_short']
    assert np.array_equal(y, x @ w)                            #(sums of at most 64 products of at most 12: exact in any order)


@pytest.mark.gpu
def test_epilogues():
    x, w, r, a, v = ints((530, 64)), ints((64, 288), -3, 4), ints((530, 288), -50, 50), ints((530, 288)), 2.0 ** ints((288,), -2, 3)
    bn     = lambda x, w, r, a, v: nn.relu((jnp.dot(x, w) - v) * v + v + r)
    two    = lambda x, w, r, a, v: (lambda c: (nn.relu(c * v), c))(jnp.dot(x, w) - v)
    steps  = lambda x, w, r, a, v: (((jnp.dot(x, w) + v) * v - r) * 0.5 + r) * v
    masked = lambda x, w, r, a, v: jnp.where(a > 0.0, jnp.dot(x, w) + r, 0.0) * v
    both   = lambda x, w, r, a, v: (lambda m: (m, m * v))(jnp.where(a > 0.0, jnp.dot(x, w), 0.0))
    for f, name in ((bn, ''), (two, ''), (steps, '_steps'), (masked, ''), (both, '')):
        with K.overrides(conv_short=True):
            _, _, fn = check_against_oracle(f, [x, w, r, a, v], exact=True)
        assert kernels_of(fn) == ['conv_gemm_split_short' + name]


def of(x, w, **choice):
    with K.overrides(**choice):
        fn = vkjax_amd.wrap(jnp.dot, frontend='minijax')
        y  = np.asarray(fn(x, w))
    kernel, = kernels_of(fn)
    assert kernel == 'conv_gemm_split_short' if 'conv_short' in choice else '_split' not in kernel, kernel
    return y


@pytest.mark.gpu
@pytest.mark.parametrize('kind', ('not finite', 'large'))
def test_sums_that_are_not_finite(kind):
    '''They are computed again with fp32 products: what those give, and the others beside them stay what they are.'''
    x, w = ints((9999, 60)), ints((60, 288), -3, 4)              #(exact in any order where they are finite)
    if kind == 'not finite':
        x[0, 3], x[40, 59], x[998, 0], x[500, 7], w[5, 287], w[9, 32] = np.inf, np.nan, -np.inf, 1e37, np.inf, np.nan
    if kind == 'large':
        x, w = x * np.float32(2.0 ** 95), w * np.float32(2.0 ** 20)         #beyond 2^80, and no partial sum (below 2^125) beyond what there is
    y, expected = of(x, w, conv_short=True), of(x, w, conv_split=False)
    same = np.isfinite(expected)
    assert np.array_equal(y[~same], expected[~same], equal_nan=True)
    assert np.array_equal(y[same], expected[same]) if kind == 'large' else np.allclose(y[same], expected[same], rtol=60 * 2.0 ** -24, atol=0)


@pytest.mark.gpu
@pytest.mark.parametrize('kind', (1, 2, 3, 4, 8, 16, 'normal', 'activations', 'small', 'all positive', 'one weight'))
@pytest.mark.parametrize('features', (36, 64))
def test_error_against_64_bits(features, kind):
    '''No larger than that of the fp32 kernels; a number: as many terms of every sum are not zero.'''
    x, w = rng.standard_normal((12000, features)).astype(np.float32), rng.standard_normal((features, 256)).astype(np.float32)
    if isinstance(kind, int):
        x *= np.argsort(rng.random_sample(x.shape), axis=1) < kind
    elif kind == 'activations':
        x = np.maximum(x, 0)
    elif kind == 'small':
        x, w = x * np.float32(1e-36), w * np.float32(1e30)
    elif kind == 'all positive':
        x, w = np.abs(x), np.abs(w)
    elif kind == 'one weight':
        w *= np.argsort(rng.random_sample(w.shape), axis=0) < 1
    exact = x.astype(np.float64) @ w.astype(np.float64)
    error = lambda y: np.linalg.norm(y - exact) / np.linalg.norm(exact)
    here, there = error(of(x, w, conv_short=True)), error(of(x, w, conv_split=False))
    print(f'{kind}, {features} features: {here:.4g}, {there:.4g}', flush=True)
    assert here <= 1.01 * there                                #(norms over 3 million results: they scatter by 0.2 %)


def test_where_they_apply():
    '''Plan only.'''
    def kernels(m, k, n, f=jnp.dot, x=None, **choice):
        zeros = lambda *s: np.broadcast_to(np.float32(0), s)
        with K.overrides(**choice):
            return [l.kernel for l in JaxprInterpreter(mj.make_jaxpr(f)(zeros(*(x or (m, k))), zeros(k, n)), plan_only=True).launches if l.kernel.startswith('conv_gemm')]
    short = lambda *a, **c: kernels(*a, **c) == ['conv_gemm_split_short']
    assert short(200704, 64, 256) and short(131072, 64, 128) and short(200704, 40, 256)
    assert not short(131071, 64, 128) and not short(200704, 32, 256) and not short(200704, 68, 256)                   #results, features
    assert not short(400000, 64, 64) and not short(200704, 64, 250)                                                    #columns
    assert not short(200704, 64, 256, conv_split='128x64') and not short(200704, 64, 256, conv_short=False) and not short(200704, 64, 256, conv_split=False)
    image = lambda stride: lambda x, w: mj.lax.conv_general_dilated(x, w.reshape((1, 1) + w.shape), (stride, stride), 'VALID', dimension_numbers=('NHWC', 'HWIO', 'NHWC'))
    assert short(0, 64, 256, f=image(1), x=(64, 56, 56, 64)) and not short(0, 64, 256, f=image(2), x=(64, 112, 112, 64))


def contract(of_lhs, of_rhs):
    return lambda x, w: mj.lax.dot_general(x, w, (((of_lhs,), (of_rhs,)), ((), ())))


def planned(f, *shapes, **choice):
    with K.overrides(**choice):
        launches = JaxprInterpreter(mj.make_jaxpr(f)(*[np.broadcast_to(np.float32(0), s) for s in shapes]), plan_only=True).launches
    return [l.kernel for l in launches if l.kernel.startswith('conv_gemm')]


@pytest.mark.parametrize('rows', (33, 40, 64))
def test_operands_contracted_over_their_rows_are_not_for_them(rows):
    '''Plan only: the kernel reads a row's features one behind the other. A dense layer's kernel gradient on so few samples, among others.'''
    gradient = mj.grad(lambda w, x: (lambda y: jnp.sum(y * y))(jnp.dot(x, w)))
    for choice in (dict(), dict(conv_short=True)):
        assert not any('short' in k for k in planned(contract(0, 0), (rows, 4096), (rows, 4096), **choice))
        assert not any('short' in k for k in planned(contract(0, 1), (rows, 4096), (4096, rows), **choice))
        assert not any('short' in k for k in planned(gradient, (4096, 4096), (rows, 4096), **choice))
    assert planned(contract(1, 1), (65536, 64), (256, 64)) == ['conv_gemm_split_short']           #(a transposed kernel operand is packed like any other)


@pytest.mark.gpu
@pytest.mark.parametrize('rows,m,n', ((64, 4096, 4096), (36, 70, 96), (64, 33, 257)))
@pytest.mark.parametrize('of_rhs', (0, 1))
def test_values_of_operands_contracted_over_their_rows(rows, m, n, of_rhs):
    x, w = ints((rows, m)), ints((rows, n), -3, 4)
    with K.overrides(**(dict() if m == 4096 else dict(conv_short=True))):
        y = np.asarray(vkjax_amd.wrap(contract(0, of_rhs), frontend='minijax')(x, w.T.copy() if of_rhs else w))
    assert np.array_equal(y, x.T @ w)                          #(exact in any order)


@pytest.mark.parametrize('k', (37, 38, 39, 61, 63))
def test_contractions_that_are_no_whole_vectors_are_not_for_them(k):
    '''Plan only.'''
    for choice in (dict(), dict(conv_short=True)):
        assert not any('short' in name for name in planned(jnp.dot, (200000, k), (k, 96), **choice))
    assert planned(jnp.dot, (200000, 40), (40, 96)) == ['conv_gemm_split_short']


@pytest.mark.gpu
@pytest.mark.parametrize('k', (33, 37, 62, 63))
def test_rows_do_not_take_from_the_next(k):
    '''Every other row is not finite, pinned to these kernels where they apply.'''
    x, w = ints((131, k)), ints((k, 96), -3, 4)
    x[1::4], x[3::4] = np.inf, np.nan
    with K.overrides(conv_short=True):
        y = np.asarray(vkjax_amd.wrap(jnp.dot, frontend='minijax')(x, w))
    assert np.array_equal(y[::2], x[::2] @ w)                  #(exact in any order)
    assert not np.isfinite(y[1::2]).any()
