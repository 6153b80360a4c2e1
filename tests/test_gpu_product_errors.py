'''Products whose sums come in another order than one block's chain over the whole contraction: shared tiles, the classes of a dilated input, kernel operands read along the
contraction or copied first. Their error against 64-bit sums is no larger than that of the general kernels, which add the contraction one step of 32 after the other.'''
import numpy as np
import pytest

import vkjax_amd
from vkjax_amd import kernels as K, minijax as mj

pytestmark = pytest.mark.gpu
lax, jnp = mj.lax, mj.numpy


def window(rhs, dilation=1, padding=((1, 1), (1, 1))):
    return lambda x, k: lax.conv_general_dilated(x, k, (1, 1), padding, lhs_dilation=(dilation, dilation), dimension_numbers=('NHWC', rhs, 'NHWC'))


def transposed(x, w):
    return lax.dot_general(x, w, (((1,), (1,)), ((), ())))


def sums(x, k):
    '''3 x 3 windows of an image with its border, in 64 bits.'''
    return sum(x[:, r:x.shape[1] - 2 + r, s:x.shape[2] - 2 + s] @ k[r, s].astype(np.float64) for r in range(3) for s in range(3))


def padded(x, dilation, padding):
    (n, h, w, c), d = x.shape, dilation
    wide = np.zeros((n, d * (h - 1) + 1, d * (w - 1) + 1, c))
    wide[:, ::d, ::d] = x
    return np.pad(wide, ((0, 0), *padding, (0, 0)))


#(program, kernel it is planned for, operands)
CASES = {'shared': (window('HWIO'), '_ks4_shared', (7, 13, 13, 256), (3, 3, 256, 256)), 'shared, another layout': (window('HWOI'), '_ks4_shared', (4, 6, 6, 256), (3, 3, 256, 256)),
         'classes': (window('HWIO', 2, ((1, 2), (1, 2))), '_ks4_strided', (7, 7, 7, 512), (3, 3, 512, 512)), 'transposed': (transposed, '_ks4t', (343, 512), (2048, 512)),
         'transposed, shared': (transposed, '_ks4t_shared', (196, 1024), (256, 1024))}


@pytest.mark.parametrize('kind', ('normal', 'activations', 'sparse'))
@pytest.mark.parametrize('name', CASES)
def test_error_against_64_bits(name, kind):
    f, kernel, xs, ws = CASES[name]
    rng  = np.random.default_rng(len(name))
    x, w = rng.standard_normal(xs).astype(np.float32), rng.standard_normal(ws).astype(np.float32)
    if kind == 'activations':
        x = np.maximum(x, 0)
    elif kind == 'sparse':
        x *= rng.random(xs) < 1 / 16
    if f is transposed:
        exact = x.astype(np.float64) @ w.T.astype(np.float64)
    elif name == 'classes':
        exact = sums(padded(x, 2, ((1, 2), (1, 2))), w)
    else:
        exact = sums(padded(x, 1, ((1, 1), (1, 1))), w.transpose(0, 1, 3, 2) if 'layout' in name else w)
    def error(wanted, **choice):
        with K.overrides(**choice):
            fn = vkjax_amd.wrap(f, frontend='minijax')
            y  = np.asarray(fn(x, w))
        kernels = [l.kernel for l in list(fn._jaxpr_interpreters.values())[0].launches if l.kernel.startswith('conv_gemm')]
        assert all(k.endswith(wanted) for k in kernels), kernels
        return np.linalg.norm(y - exact) / np.linalg.norm(exact)
    here, there = error(kernel), error('', conv_ksplit=False, conv_tile='64x64', conv_bk=32)
    print(f'{name}, {kind}: {here:.4g}, {there:.4g}', flush=True)
    assert here <= 1.01 * there
