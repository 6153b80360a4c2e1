'''Kernel operands of other layouts are copied into the dense one (K.dense_copy_pays) where more than one tile of rows reads them.'''
import numpy as np
import pytest

import vkjax_amd
from vkjax_amd import minijax as mj
from vkjax_amd.jaxpr_interpreter import JaxprInterpreter

lax = mj.lax


def transposed(x, w):
    return lax.dot_general(x, w, (((1,), (1,)), ((), ())))


def window(x, w):
    return lax.conv_general_dilated(x, w, (1, 1), ((1, 1), (1, 1)), dimension_numbers=('NHWC', 'HWOI', 'NHWC'))


def copies(f, *shapes):
    program = JaxprInterpreter(mj.make_jaxpr(f)(*[np.broadcast_to(np.float32(0), s) for s in shapes]), plan_only=True)
    return any(l.kernel.startswith('transpose_tiled') for l in program.launches)


@pytest.mark.parametrize('m,k,n,copied', [(1, 2048, 50000, False), (32, 768, 30524, False), (8, 1024, 128000, False), (64, 768, 30524, False),
                                          (64, 512, 20000, True), (65, 768, 30524, True), (128, 4096, 16384, True), (1024, 512, 20000, True),
                                          (1, 2048, 30000, False), (32, 512, 66000, False)])
def test_operands_that_few_rows_read_are_not_copied(m, k, n, copied):
    '''Plan only.'''
    assert copies(transposed, (m, k), (n, k)) == copied


@pytest.mark.parametrize('size,c,n,copied', [(2, 2048, 2048, False), (4, 1024, 1024, True), (4, 1024, 2048, False), (7, 512, 512, True), (7, 512, 4096, True)])
def test_kernels_of_windows(size, c, n, copied):
    '''Plan only.'''
    assert copies(window, (1, size, size, c), (3, 3, n, c)) == copied


@pytest.mark.gpu
@pytest.mark.parametrize('m,k,n', [(1, 516, 33000), (32, 512, 33000), (33, 516, 20000), (64, 512, 33000), (65, 512, 33000)])
def test_values_on_both_sides_of_the_line(m, k, n):
    rng = np.random.default_rng(m)
    x, w = (rng.integers(-4, 5, size=s).astype(np.float32) for s in ((m, k), (n, k)))
    assert np.array_equal(np.asarray(vkjax_amd.wrap(transposed, frontend='minijax')(x, w)), x @ w.T)      #(exact in any order)
