'''Products whose 32 x 32 tiles several blocks share: each sums a slice of the contraction, the last to arrive adds the slices.'''
import numpy as np
import pytest

import vkjax_amd
from vkjax_amd import kernels as K, minijax as mj
from vkjax_amd.minijax import tree_util
from tests.common import check_against_oracle

lax, nn, jnp = mj.lax, mj.nn, mj.numpy
DN = ('NHWC', 'HWIO', 'NHWC')


def conv(x, w):
    return lax.conv_general_dilated(x, w, (1, 1), 'SAME', dimension_numbers=DN)


def plain(x, w):
    return jnp.dot(x, w)


def residual(x, w, mean, scale, beta, rest):
    return nn.relu((conv(x, w) - mean) * scale + beta + rest)


def both(x, w, mean, scale):
    centred = conv(x, w) - mean
    return centred, nn.relu(centred * scale)


def clipped(x, w, mean):
    return jnp.minimum(nn.relu(conv(x, w) - mean), np.float32(6))


def launches_of(fn):
    return list(fn._jaxpr_interpreters.values())[0].launches


def integers(f, shape_x, shape_w, seed=3):
    rng  = np.random.RandomState(seed)
    ints = lambda lo, hi, *s: rng.randint(lo, hi, size=s).astype(np.float32)
    n    = shape_w[-1]
    rest = {plain: [], residual: [ints(-5, 5, n), ints(1, 4, n), ints(-9, 9, n), ints(-50, 50, *shape_x[:-1], n)], both: [ints(-5, 5, n), ints(1, 4, n)],
            clipped: [ints(-5, 5, n)]}[f]
    return [ints(-4, 5, *shape_x), ints(-3, 4, *shape_w)] + rest


#ragged rows and columns, contractions that end within a step, slices of unequal length, later slices that start at another tap; an odd number of columns
#takes word loads of the kernel operand. The share that is asked for and the number of blocks it comes to
CASES = [(plain, (33, 900), (900, 36), 2, 2), (plain, (70, 1300), (1300, 7 + 32), 3, 3), (plain, (129, 388), (388, 100), 8, 4), (plain, (1, 1156), (1156, 64), 7, 5),
         (residual, (1, 7, 7, 128), (3, 3, 128, 40), 4, 3), (residual, (2, 5, 6, 256), (3, 3, 256, 33), 8, 6), (residual, (1, 9, 7, 512), (1, 1, 512, 72), 2, 2),
         (both, (1, 14, 14, 256), (3, 3, 256, 64), 5, 5), (clipped, (1, 9, 9, 256), (3, 3, 256, 64), 3, 3)]


@pytest.mark.gpu
@pytest.mark.parametrize('general', (False, True))
@pytest.mark.parametrize('f,x,w,shares,blocks', CASES)
def test_integers_are_exact(f, x, w, shares, blocks, general):
    print('shared tiles:', f.__name__, x, w, shares, general, flush=True)
    args = integers(f, x, w)
    with K.overrides(conv_ksplit=True, conv_shares=shares, conv_k_splits=1, conv_b_general=general):
        _, ytrue, fn = check_against_oracle(f, args, exact=True)
    product, *others = launches_of(fn)
    m = int(np.prod(x[:-1]))
    assert product.kernel == f'conv_gemm_32x32x128_ks4{"g" if general else ""}_shared' and product.grid[0] == -(-m // 32) * -(-w[-1] // 32) * blocks
    assert len(others) == (f is clipped)
    for _ in range(3):                                            #the counters are zero again
        for got, want in zip(tree_util.tree_leaves(fn(*args)), tree_util.tree_leaves(ytrue)):
            assert np.array_equal(got, want)


@pytest.mark.gpu
@pytest.mark.parametrize('batch,size,cin,cout,window', [(1, 28, 128, 128, 3), (1, 14, 1024, 256, 1), (4, 7, 512, 512, 3), (7, 7, 512, 512, 3), (12, 7, 2048, 512, 1)])
def test_values_by_the_estimate(batch, size, cin, cout, window):
    print('shared by the estimate:', batch, size, cin, cout, window, flush=True)
    rng  = np.random.default_rng(batch + cin)
    x, w = rng.standard_normal((batch, size, size, cin)).astype(np.float32), rng.standard_normal((window, window, cin, cout)).astype(np.float32)
    fn   = vkjax_amd.wrap(conv, frontend='minijax')
    got  = fn(x, w)
    assert launches_of(fn)[0].kernel == 'conv_gemm_32x32x128_ks4_shared' and len(launches_of(fn)) == 1
    padded = np.pad(x.astype(np.float64), ((0, 0), (window // 2,) * 2, (window // 2,) * 2, (0, 0)))
    shifted = [(padded[:, r:r + size, s:s + size].reshape(-1, cin), w[r, s].astype(np.float64)) for r in range(window) for s in range(window)]
    exact, reach = sum(a @ b for a, b in shifted), sum(np.abs(a) @ np.abs(b) for a, b in shifted)
    #as many roundings of the sum of the magnitudes as there are products
    assert np.all(np.abs(got.reshape(-1, cout) - exact) <= window * window * cin * 2.0**-24 * reach)


def test_share_counts():
    '''One block per tile where that fills the CUs or the contraction is short; never more blocks than steps.'''
    assert [K.choose_conv_shares(*a) for a in ((100, 4), (128, 4), (200, 18), (200, 8), (400, 16), (2048, 36), (400, 36))] == [1] * 7
    assert all(1 < K.choose_conv_shares(*a) <= min(a[1], K.CONV_MAX_SHARES) for a in ((56, 18), (56, 8), (100, 9), (104, 18), (112, 36), (160, 36), (304, 36)))


def test_what_shared_tiles_need_is_refused_otherwise():
    '''With the error that callers who try a part of a product expect, who then launch the whole of it.'''
    buffer = lambda *shape: K.Buffer(None, np.dtype(np.float32), shape)
    out, lhs, rhs = buffer(70, 40), buffer(70, 1026), buffer(1026, 40)
    geom = K.ConvGeometry(batch=1, Ho=70, Wo=1, N=40, H=70, W=1, Cin=1026, KH=1, KW=1, xs=(0, 1026, 0, 1), ws=(1026 * 40, 1026 * 40, 40, 1), os=(70 * 40, 40, 40, 1))
    with K.overrides(conv_ksplit=True):
        def launch(count=3, partial=3 * 6 * 1024, arrivals=K.CONV_MAX_SHARED_TILES, **offsets):
            return K.conv_gemm(out, lhs, rhs, geom._replace(shares=K.ConvShares(count, buffer(partial), buffer(arrivals))), **offsets)
        assert launch().kernel == 'conv_gemm_32x32x128_ks4_shared'
        for wrong in (dict(out_offset=4), dict(count=7, partial=7 * 6 * 1024), dict(arrivals=5), dict(partial=3 * 6 * 1024 - 1)):
            with pytest.raises(ValueError):
                launch(**wrong)
