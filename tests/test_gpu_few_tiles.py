'''Products of few 32 x 32 tiles on both sides of the lines up to which four waves share a tile: the kernel that is chosen, and
64-bit values within fp32's reach.'''
import numpy as np
import pytest

import vkjax_amd
from vkjax_amd import minijax as mj
from vkjax_amd.minijax import lax


def layer(x, w, shift, rest):
    return mj.nn.relu(mj.numpy.dot(x, w) + shift + rest)


def layer_transposed(x, w, shift, rest):
    return mj.nn.relu(lax.dot_general(x, w, (((1,), (1,)), ((), ()))) + shift + rest)


#(M, K, N, kernel operand transposed, four waves per tile): one, two, three, four and five rounds of a tile per CU; contractions shorter
#than a step of 128, of whole steps, and with a remainder of one vector; ragged rows and columns
CASES = [(33, 4, 36, 0, 1), (1000, 32, 100, 0, 1), (196, 68, 512, 0, 1), (255, 124, 1020, 0, 1), (513, 60, 512, 0, 0), (513, 64, 512, 0, 1), (784, 132, 510, 0, 1),
         (256, 252, 2044, 0, 1), (545, 124, 992, 0, 1), (545, 96, 992, 0, 0), (784, 192, 768, 0, 0), (784, 320, 766, 0, 1), (784, 512, 1000, 0, 0), (1024, 1024, 1022, 0, 1),
         (1025, 1024, 1022, 0, 0), (64, 60, 100, 1, 0), (200, 64, 1000, 1, 1), (255, 100, 2048, 1, 0), (255, 128, 2044, 1, 1), (250, 200, 2100, 1, 0)]


def arguments(M, K, N, transposed):
    rng = np.random.default_rng(M + K + N)
    return [rng.standard_normal(s).astype(np.float32) for s in ((M, K), (N, K) if transposed else (K, N), (N,), (M, N))]


@pytest.mark.parametrize('M,K,N,transposed,four', CASES)
def test_kernel_chosen(M, K, N, transposed, four):
    args = arguments(M, K, N, transposed)
    interp, _ = vkjax_amd.wrap(layer_transposed if transposed else layer, frontend='minijax', plan_only=True)._get_or_create_jaxpr_interpreter(args)
    product,  = [l.kernel for l in interp.launches if l.kernel.startswith('conv_gemm')]
    assert ('_ks4' in product) == bool(four), product


@pytest.mark.gpu
@pytest.mark.parametrize('M,K,N,transposed,four', CASES)
def test_values(M, K, N, transposed, four):
    print('product', M, K, N, transposed, flush=True)
    args = x, w, shift, rest = arguments(M, K, N, transposed)
    w64  = (w.T if transposed else w).astype(np.float64)
    got  = vkjax_amd.wrap(layer_transposed if transposed else layer, frontend='minijax')(*args)
    exact = np.maximum(x.astype(np.float64) @ w64 + shift + rest, 0)
    #K products and three more sums in fp32: at most as many roundings of the sum of the magnitudes
    bound = (K + 3) * 2.0**-24 * (np.abs(x).astype(np.float64) @ np.abs(w64) + np.abs(shift) + np.abs(rest))
    assert np.all(np.abs(got - exact) <= bound)
