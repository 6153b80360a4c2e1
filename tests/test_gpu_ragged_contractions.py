'''Products whose contraction is no multiple of four: rows that begin at any word, and a last vector that reads into the next row.'''
import numpy as np
import pytest

import vkjax_amd
from vkjax_amd import kernels as K, minijax as mj
from vkjax_amd.jaxpr_interpreter import JaxprInterpreter

lax, nn, jnp = mj.lax, mj.nn, mj.numpy


def layer(x, w, b):
    return nn.relu(jnp.dot(x, w) + b)


def inputs(M, Kc, N):
    rng = np.random.default_rng(M + 7 * Kc + N)
    return [rng.standard_normal(s).astype(np.float32) for s in ((M, Kc), (Kc, N), (N,))]


def kernel(f, args, **choices):
    with K.overrides(**choices):
        return JaxprInterpreter(mj.make_jaxpr(f)(*args), plan_only=True).launches[0].kernel


#(kernel, M, K, N, pinned): contractions of less than a vector, of one to three words beyond whole vectors, steps and slices; each of the kernels with 16-byte loads of the rows
CASES = [('dense_rows_n16', 9, 1, 7, {}), ('dense_rows_n16', 33, 255, 12, {}), ('dense_rows_n16', 33, 513, 16, {}), ('dense_rows_n16', 5, 1026, 3, {}),
         ('conv_gemm_32x32x128_ks4', 33, 3, 36, {}), ('conv_gemm_32x32x128_ks4', 65, 127, 40, {}), ('conv_gemm_32x32x128_ks4', 40, 385, 33, {}),
         ('conv_gemm_32x32x128_ks4', 31, 1301, 24, dict(conv_k_splits=3)), ('conv_gemm_32x32x128_ks4_shared', 70, 1026, 40, dict(conv_ksplit=True, conv_shares=4, conv_k_splits=1)),
         ('conv_gemm_32x32x128_ks4g', 40, 259, 36, dict(conv_b_general=True, conv_ksplit=True)), ('conv_gemm_64x64x32_lean', 70, 97, 72, dict(conv_tile='64x64', conv_bk=32)),
         ('conv_gemm_64x64x64_lean', 70, 130, 72, dict(conv_tile='64x64', conv_bk=64)), ('conv_gemm_32x32x32_lean', 70, 61, 72, dict(conv_tile='32x32', conv_bk=32)),
         ('conv_gemm_64x64x32_fg', 70, 67, 71, dict(conv_tile='64x64', conv_bk=32, conv_b_general=True)), ('conv_gemm_64x64x32_mix', 200, 261, 72, dict(conv_mix=2, conv_tile='64x64', conv_bk=32))]


@pytest.mark.parametrize('name,M,Kc,N,choices', CASES)
def test_kernel_chosen(name, M, Kc, N, choices):
    assert kernel(layer, inputs(M, Kc, N), **choices) == name


@pytest.mark.gpu
@pytest.mark.parametrize('name,M,Kc,N,choices', CASES)
def test_values(name, M, Kc, N, choices):
    print('ragged contraction:', name, M, Kc, N, flush=True)
    args = x, w, b = inputs(M, Kc, N)
    with K.overrides(**choices):
        fn = vkjax_amd.wrap(layer, frontend='minijax')
        got = fn(*args)
        exact = np.maximum(x.astype(np.float64) @ w.astype(np.float64) + b, 0)
        #K products and two more sums in fp32: at most as many roundings of the sum of the magnitudes
        bound = (Kc + 2) * 2.0**-24 * (np.abs(x).astype(np.float64) @ np.abs(w).astype(np.float64) + np.abs(b))
        assert np.all(np.abs(got - exact) <= bound)
        #what follows a row's last value is not seen: every other row infinite or NaN
        for odd in (np.inf, np.nan):
            x[1::2] = odd
            again = fn(x, w, b)
            assert np.array_equal(again[::2], got[::2])


@pytest.mark.gpu
def test_strided_pixels_of_an_odd_number_of_features():
    '''A 1 x 1 window at a stride of 2: rows are not consecutive.'''
    rng  = np.random.default_rng(5)
    x, w = rng.integers(-4, 5, size=(2, 9, 7, 131)).astype(np.float32), rng.integers(-3, 4, size=(1, 1, 131, 45)).astype(np.float32)
    f    = lambda x, w: lax.conv_general_dilated(x, w, (2, 2), 'SAME', dimension_numbers=('NHWC', 'HWIO', 'NHWC'))
    assert kernel(f, [x, w]) == 'conv_gemm_32x32x128_ks4'
    assert np.array_equal(vkjax_amd.wrap(f, frontend='minijax')(x, w), x[:, ::2, ::2].reshape(-1, 131).dot(w[0, 0]).reshape(2, 5, 4, 45))


def test_many_rows_of_few_features_go_to_tiles():
    shapes = [(2048, 257, 10), (2049, 257, 10), (1280, 510, 16), (1281, 510, 16), (100000, 256, 10)]
    assert ['dense' in kernel(layer, [np.zeros(s, np.float32) for s in ((m, k), (k, n), (n,))]) for m, k, n in shapes] == [True, False, True, False, True]


def test_short_contractions_keep_their_epilogue():
    '''Plan only: a residual behind a product of few odd features is part of its launch.'''
    f    = lambda x, w, b, r: nn.relu(jnp.dot(x, w) + b + r)
    plan = lambda m, k, n: [l.kernel for l in JaxprInterpreter(mj.make_jaxpr(f)(*[np.zeros(s, np.float32) for s in ((m, k), (k, n), (n,), (m, n))]), plan_only=True).launches]
    for m, k, n in ((551, 25, 16), (3910, 13, 4), (61, 9, 16), (359, 17, 13), (50, 31, 8)):
        assert len(plan(m, k, n)) == 1 and 'dense' not in plan(m, k, n)[0], (m, k, n)
    assert plan(50, 33, 8)[0] == 'dense_rows_n16' and plan(50, 28, 8)[0] == 'dense_rows_n16'


def test_large_full_tensors_behind_one_step():
    f    = lambda x, w, b, r: nn.relu(jnp.dot(x, w) + b + r)
    zero = lambda *s: np.broadcast_to(np.float32(0), s)
    plan = lambda m, k, n: JaxprInterpreter(mj.make_jaxpr(f)(zero(m, k), zero(k, n), zero(n), zero(m, n)), plan_only=True).launches[0].kernel
    for m, k, n, kernel in ((255921, 13, 104, 'gf'), (24088, 5, 256, 'gf'), (255921, 12, 104, 'lean'), (179393, 33, 64, 'lean'), (40426, 6, 104, 'lean')):
        assert plan(m, k, n).endswith('_' + kernel), (m, k, n, plan(m, k, n))


@pytest.mark.gpu
def test_values_of_large_full_tensors_behind_one_step():
    rng = np.random.default_rng(8)
    x, w, b, r = (rng.integers(-4, 5, size=s).astype(np.float32) for s in ((60001, 7), (7, 90), (90,), (60001, 90)))
    assert np.array_equal(vkjax_amd.wrap(lambda x, w, b, r: nn.relu(jnp.dot(x, w) + b + r), frontend='minijax')(x, w, b, r), np.maximum(x @ w + b + r, 0))
