'''Convolutions of images of very few features (conv_gemm_stem_*): images that tiles do not divide, rows that are no whole vectors, tiles that reach into many
image rows, a handful of positions. Whole numbers, so every result is exact.'''
import numpy as np
import pytest

from vkjax_amd import kernels as K, minijax as mj
from tests.common import check_against_oracle

lax, nn = mj.lax, mj.nn
rng = np.random.RandomState(23)


def ints(lo, hi, *s):
    return rng.randint(lo, hi, size=s).astype(np.float32)


#(images, height, width), features out, strides, padding
SIZES = [((2, 24, 25), 64, (2, 2), ((3, 3), (3, 3))), ((3, 9, 9), 33, (1, 1), ((1, 1), (1, 1))), ((1, 40, 101), 64, (2, 2), ((0, 0), (0, 0))), ((2, 13, 200), 8, (2, 1), ((3, 2), (2, 5))),
         ((1, 9, 9), 5, (2, 2), ((0, 0), (0, 0))), ((2, 33, 31), 64, (3, 2), ((2, 3), (0, 1))), ((1, 67, 17), 40, (1, 1), ((3, 3), (3, 3))), ((5, 16, 16), 64, (2, 2), ((3, 3), (3, 3)))]


@pytest.mark.gpu
@pytest.mark.parametrize('window,tile', ((7, True), (7, 64), (3, True)))
@pytest.mark.parametrize('images,features,strides,padding', SIZES)
def test_sizes(images, features, strides, padding, window, tile):
    print('stem:', images, features, strides, padding, window, tile, flush=True)
    def f(x, w, mean, scale, beta):
        y = lax.conv_general_dilated(x, w, strides, padding, dimension_numbers=('NHWC', 'HWIO', 'NHWC')) - mean
        return y, nn.relu(y * scale + beta)
    args = [ints(-4, 5, *images, 3), ints(-3, 4, window, window, 3, features), ints(-5, 5, features), ints(1, 4, features), ints(-9, 9, features)]
    with K.overrides(conv_stem=tile):
        _, ytrue, fn = check_against_oracle(f, args, exact=True)
        for a, b in zip(fn(*args), ytrue):                         #a second pass: other tiles were in LDS last
            assert np.array_equal(a, b)
    kernels = [l.kernel for l in list(fn._jaxpr_interpreters.values())[0].launches]
    assert kernels[0] == {7: {True: 'conv_gemm_stem_7x22_m128', 64: 'conv_gemm_stem_7x22'}[tile], 3: 'conv_gemm_stem_3x10_m128'}[window], kernels


def test_patches_that_do_not_fit():
    '''Image rows too long for the patch are left to the other kernels.'''
    import vkjax_amd
    def f(x, w):
        return lax.conv_general_dilated(x, w, (1, 1), 'SAME', dimension_numbers=('NHWC', 'HWIO', 'NHWC'))
    for width, stem in ((200, True), (1000, False)):
        interp, _ = vkjax_amd.wrap(f, frontend='minijax', plan_only=True)._get_or_create_jaxpr_interpreter([ints(-1, 2, 1, 20, width, 3), ints(-1, 2, 7, 7, 3, 16)])
        assert interp.launches[-1].kernel.startswith('conv_gemm_stem') == stem, interp.launches[-1].kernel


@pytest.mark.parametrize('window,stride,images,size,features,stem', [
    (7, 2, 1, 64, 8, True), (7, 2, 64, 224, 64, True), (7, 2, 9, 209, 4, True), (7, 2, 200, 24, 64, True), (7, 2, 100, 9, 64, True),
    (7, 2, 300, 9, 64, False), (7, 2, 2000, 9, 64, False), (7, 2, 1000, 16, 8, False),
    (3, 2, 50, 97, 64, True), (3, 2, 50, 97, 33, True), (3, 2, 50, 97, 32, False), (3, 2, 64, 224, 8, False), (3, 1, 90, 32, 64, True), (3, 1, 120, 32, 40, True),
    (3, 2, 20, 141, 64, False), (3, 1, 2000, 9, 64, False), (3, 1, 1100, 8, 64, False), (3, 1, 300, 17, 64, False), (3, 2, 200, 41, 64, False)])
def test_where_they_pay(window, stride, images, size, features, stem):
    '''Plan only: few features, or images that fill their tiles badly, are left to the general kernel.'''
    from vkjax_amd.jaxpr_interpreter import JaxprInterpreter
    p = window // 2
    def f(x, w):
        return lax.conv_general_dilated(x, w, (stride, stride), ((p, p), (p, p)), dimension_numbers=('NHWC', 'HWIO', 'NHWC'))
    zeros  = lambda *s: np.broadcast_to(np.float32(0), s)
    launch = JaxprInterpreter(mj.make_jaxpr(f)(zeros(images, size, size, 3), zeros(window, window, 3, features)), plan_only=True).launches[-1]
    assert launch.kernel.startswith('conv_gemm_stem') == stem, launch.kernel
