'''The backward pass of a ReLU as the epilogue of a product on the bf16 matrix cores (CONV_MASK): + full tensor, mask by an activation,
second result, * vector. The arithmetic is that of the launches it replaces, so integer-valued data give equal results.'''
import numpy as np
import pytest

from vkjax_amd import kernels as K
from vkjax_amd import minijax as mj
from vkjax_amd.jaxpr_interpreter import JaxprInterpreter

from .common import check_against_oracle

lax, jnp, nn = mj.lax, mj.numpy, mj.nn
DN = ('NHWC', 'HWIO', 'NHWC')
rng = np.random.RandomState(37)


def ints(shape, low=-4, high=5):
    return rng.randint(low, high, size=shape).astype(np.float32)


def product(g, w):
    return lax.conv_general_dilated(g, w, (1, 1), 'SAME', dimension_numbers=DN)

def masked(g, w, act, r, k):
    return jnp.where(act > 0, product(g, w), 0.0)
def masked_scaled(g, w, act, r, k):
    return jnp.where(act > 0, product(g, w), 0.0) * k
def added_masked(g, w, act, r, k):
    return jnp.where(act > 0.5, product(g, w) + r, -2.0)
def added_masked_scaled(g, w, act, r, k):
    return jnp.where(act > 0, product(g, w) + r, 0.0) * k
def both(g, w, act, r, k):
    m = jnp.where(act > 0, product(g, w) + r, 0.0)
    return m, m * k
def both_later(g, w, act, r, k):
    m = jnp.where(act > 0, product(g, w), 0.0)
    return m * (k + 1.0), m
def two_scalings(g, w, act, r, k):
    m = jnp.where(act > 0, product(g, w) + r, 0.0)
    return m * k, k * m + r

def vector_of_the_result(g, w, act, r, k):                #known behind the mask only: the product stays a launch of its own
    m = jnp.where(act > 0, product(g, w), 0.0)
    return m * jnp.sum(m, axis=(0, 1, 2))

FUSED     = [masked, masked_scaled, added_masked, added_masked_scaled, both, both_later, two_scalings, vector_of_the_result]

def product_used_twice(g, w, act, r, k):
    d = product(g, w)
    return jnp.where(act > 0, d, 0.0), d
def kept_where_not_above(g, w, act, r, k):
    return jnp.where(act > 0, 0.0, product(g, w))
def masked_by_itself(g, w, act, r, k):
    d = product(g, w)
    return jnp.where(d > 0, d, 0.0)

OTHERS    = [product_used_twice, kept_where_not_above, masked_by_itself]

#(rows around a tile's 128, columns around 64 and 128; 1x1 and 3x3)
SHAPES = [([1, 127, 1, 32], [1, 1, 32, 63]), ([2, 9, 15, 32], [3, 3, 32, 132]), ([1, 16, 8, 64], [1, 1, 64, 128])]


def arguments(xs, ks):
    shape = xs[:3] + [ks[3]]
    return [ints(xs), ints(ks, -3, 4), ints(shape, -2, 3), ints(shape, -50, 51), ints([ks[3]], -3, 4)]


def masks(launches):
    return [l for l in launches if l.kernel.startswith('conv_gemm_split') and np.frombuffer(l.params, np.uint32)[21] >> 25 & 1]


@pytest.mark.gpu
@pytest.mark.parametrize('tile', list(K.CONV_SPLIT_TILES))
@pytest.mark.parametrize('f', FUSED + OTHERS, ids=lambda f: f.__name__)
def test_results(f, tile):
    for xs, ks in SHAPES:
        for slices in (1, 3):
            if slices > 1 and 2 * -(-int(np.prod(ks[:3])) // 64) < 2 * slices:
                continue
            print(f'case: {f.__name__}, tile {tile}, {slices} slices, {xs} {ks}', flush=True)
            with K.overrides(conv_split=tile, conv_split_slices=slices):
                _, _, fn = check_against_oracle(f, arguments(xs, ks), exact=True)
            assert len(masks(list(fn._jaxpr_interpreters.values())[0].launches)) == (f in FUSED)


@pytest.mark.gpu
def test_values_that_are_not_finite():
    '''A NaN in the activation is not above the limit; products that are infinite or NaN pass where it is.'''
    g, w, act, r, k = arguments([1, 140, 1, 32], [1, 1, 32, 70])
    act[0, 3, 0, 5], act[0, 130, 0, 69], act[0, 7, 0, :] = np.nan, np.inf, -np.inf
    g[0, 9, 0, 1], g[0, 133, 0, 31], r[0, 3, 0, 5], r[0, 20, 0, 0] = np.inf, np.nan, np.nan, np.inf
    for f in (masked_scaled, both):
        with K.overrides(conv_split=True):
            check_against_oracle(f, [g, w, act, r, k], exact=True)


@pytest.mark.parametrize('f', FUSED + OTHERS, ids=lambda f: f.__name__)
def test_which_programs_are_merged(f):
    '''Plan only: one launch for all of it where the pattern holds, and its operands at their places; else the launches as they were.'''
    args = arguments([1, 16, 8, 64], [1, 1, 64, 128])
    with K.overrides(conv_split=True):
        program = JaxprInterpreter(mj.make_jaxpr(f)(*args), plan_only=True)
    merged = masks(program.launches)
    assert len(merged) == (f in FUSED)
    if f is both:
        buffers = [b for b, _ in merged[0].buffers]
        m, dx = program.output_buffers
        assert buffers[0] is dx and buffers[5 + K.CONV_MAX_EPI - 1] is m and len(program.launches) == 2          #the packing and the product
        assert all(buffers[5 + i]._placeholder is program.input_buffers[j]._placeholder for i, j in enumerate((3, 2, 4)))
    if f is vector_of_the_result:
        assert merged[0].buffers[7][0] is None and merged[0].buffers[5 + K.CONV_MAX_EPI - 1][0] is None
