'''The kernel-gradient kernels on the bf16 matrix cores (csrc/kernels/wgrad_split.h). Integer-valued data make every product and sum
exact, so those results have to be equal whatever the slices; on random data the error against 64-bit sums is compared with that of
the fp32 kernels, which it must not exceed.'''
import numpy as np
import pytest

import vkjax_amd
from vkjax_amd import kernels as K
from vkjax_amd import minijax as mj
from vkjax_amd.jaxpr_interpreter import JaxprInterpreter

from .common import check_against_oracle

lax, jnp = mj.lax, mj.numpy
DN = ('NHWC', 'HWIO', 'NHWC')
rng = np.random.RandomState(29)


def kernel_gradient(strides=(1, 1), padding=((0, 0), (0, 0)), dilation=(1, 1)):
    def loss(x, w, g):
        return jnp.sum(lax.conv_general_dilated(x, w, strides, padding, rhs_dilation=dilation, dimension_numbers=DN) * g)
    return lambda x, w, g: mj.grad(loss, argnums=1)(x, w, g)


def product(x, g):
    return lax.dot_general(x, g, (((0,), (0,)), ((), ())))


def wgrads(launches):
    return [l for l in launches if l.kernel.startswith('wgrad')]


P1 = ((1, 1), (1, 1))
#rows and columns of the result around the tiles' edges, contractions that end inside a k tile, a slice or an octet; taps outside
#the image, strides, dilation, crops; features that 16-byte loads cannot take
SHAPES = [   #x, kernel, G's (y, x), strides, padding, dilation
    ('64 x 64',               (2, 12, 11, 64), (1, 1, 64, 64),  (12, 11), (1, 1), ((0, 0), (0, 0)), (1, 1)),
    ('4 x 4',                 (1, 16, 9, 4),   (1, 1, 4, 4),    (16, 9),  (1, 1), ((0, 0), (0, 0)), (1, 1)),
    ('132 x 60',              (3, 7, 7, 132),  (1, 1, 132, 60), (7, 7),   (1, 1), ((0, 0), (0, 0)), (1, 1)),
    ('3x3',                   (3, 8, 9, 20),   (3, 3, 20, 132), (8, 9),   (1, 1), P1, (1, 1)),
    ('3x3 stride 2',          (4, 13, 11, 8),  (3, 3, 8, 68),   (7, 6),   (2, 2), P1, (1, 1)),
    ('1x1 stride 2',          (4, 15, 14, 12), (1, 1, 12, 36),  (8, 7),   (2, 2), ((0, 0), (0, 0)), (1, 1)),
    ('dilated, uneven pads',  (2, 13, 14, 16), (3, 2, 16, 8),   (12, 12), (1, 1), ((3, 0), (0, 1)), (2, 3)),
    ('crop',                  (2, 13, 14, 16), (1, 1, 16, 8),   (10, 11), (1, 1), ((-1, -2), (-3, 0)), (1, 1)),
    ('3 features',            (2, 20, 21, 3),  (7, 7, 3, 64),   (10, 11), (2, 2), ((3, 3), (3, 3)), (1, 1)),
    ('5 features',            (2, 9, 9, 5),    (3, 3, 5, 12),   (9, 9),   (1, 1), P1, (1, 1)),
]


@pytest.mark.gpu
@pytest.mark.parametrize('tile', list(K.WGRAD_SPLIT_TILES))
@pytest.mark.parametrize('desc,xs,ws,gyx,strides,padding,dilation', SHAPES, ids=[s[0] for s in SHAPES])
def test_tile_edges_and_slices(tile, desc, xs, ws, gyx, strides, padding, dilation):
    x, w = rng.randint(-4, 5, size=xs).astype(np.float32), np.zeros(ws, np.float32)
    g = rng.randint(-3, 4, size=(xs[0],) + gyx + ws[3:]).astype(np.float32)
    for slices in (1, 2, 3, 1000):
        print(f'case: {desc}, tile {tile}, {slices} slices', flush=True)
        with K.overrides(wgrad_split=tile, wgrad_slices=slices):
            _, _, fn = check_against_oracle(kernel_gradient(strides, padding, dilation), [x, w, g], exact=True)
        kernels = [l.kernel for l in wgrads(list(fn._jaxpr_interpreters.values())[0].launches)]
        loads = 'a' if xs[3] % 4 == 0 else 's'
        assert kernels == [f'wgrad_split_{tile}_{loads}a' if loads in K.WGRAD_SPLIT_TILES[tile][4] else 'wgrad_gemm_64x64_sa'], kernels


@pytest.mark.gpu
@pytest.mark.parametrize('desc,xs,ws,gyx,strides,padding,dilation', SHAPES, ids=[s[0] for s in SHAPES])
def test_sums_computed_again_with_fp32_products(desc, xs, ws, gyx, strides, padding, dilation):
    '''Over the same shapes, with operands that are not finite in X and G.'''
    x, w = rng.randint(-4, 5, size=xs).astype(np.float32), np.zeros(ws, np.float32)
    g = rng.randint(-3, 4, size=(xs[0],) + gyx + ws[3:]).astype(np.float32)
    x.reshape(-1)[rng.permutation(x.size)[:3]] = np.inf, np.nan, -np.inf
    g.reshape(-1)[rng.permutation(g.size)[:2]] = np.inf, -np.inf
    f = kernel_gradient(strides, padding, dilation)
    results = {}
    for tile in list(K.WGRAD_SPLIT_TILES) + [False]:
        for slices in (1, 3):
            print(f'case: {desc}, tile {tile}, {slices} slices', flush=True)
            with K.overrides(wgrad_split=tile, wgrad_slices=slices):
                results[tile, slices] = vkjax_amd.wrap(f, frontend='minijax')(x, w, g)
    expected = results[False, 1]
    assert not np.isfinite(expected).all() and all(np.array_equal(y, expected, equal_nan=True) for y in results.values())


@pytest.mark.gpu
@pytest.mark.parametrize('pixels,M,N', [(200, 40, 72), (2049, 132, 128), (12544, 256, 64)])
def test_error_against_64_bit_sums_is_no_larger(pixels, M, N):
    x, g = rng.standard_normal((pixels, M)).astype(np.float32), rng.standard_normal((pixels, N)).astype(np.float32)
    exact = x.astype(np.float64).T @ g.astype(np.float64)
    def error(**choice):
        with K.overrides(**choice):
            fn = vkjax_amd.wrap(product, frontend='minijax')
            y = fn(x, g)
        return np.linalg.norm(y - exact) / np.linalg.norm(exact)
    fp32 = error(wgrad_split=False)
    for tile in K.WGRAD_SPLIT_TILES:
        e = error(wgrad_split=tile)
        print(f'{pixels} x {M} x {N}, tile {tile}: {e:.2e}, fp32 products {fp32:.2e}', flush=True)
        assert e <= fp32


@pytest.mark.gpu
@pytest.mark.parametrize('value', (np.inf, -np.inf, np.nan, 3.4e38, -3.4e38, 1e-30))
def test_values_a_bf16_part_cannot_hold(value):
    '''An infinity, a NaN and numbers beyond the largest bf16 leave what fp32 products leave; the rest of the result is not touched.'''
    x, g = rng.randint(1, 4, size=(320, 136)).astype(np.float32), rng.randint(1, 4, size=(320, 72)).astype(np.float32) * np.float32(2.0**-8)
    x[301, 130] = value
    exact = (x.astype(np.float64)[:, :, None] * g.astype(np.float64)[:, None, :]).sum(0) if np.isfinite(value) else None
    for tile in K.WGRAD_SPLIT_TILES:
        with K.overrides(wgrad_split=tile, wgrad_slices=3):
            y = vkjax_amd.wrap(product, frontend='minijax')(x, g)
        if exact is None:
            assert (np.isnan(y[130]) if np.isnan(value) else y[130] == value).all()
        else:
            assert np.allclose(y[130], exact[130], rtol=320 * 2.0**-24)       #one rounding per term
        rest = np.arange(136) != 130
        assert np.array_equal(y[rest], (x[:, rest].T.astype(np.float64) @ g.astype(np.float64)).astype(np.float32))


def test_which_gradients_take_the_kernels():
    '''The rule: enough operations, G's features in fours, an image whose coordinates fit 16 bits.'''
    G = K.WgradGeometry
    layer = lambda **k: G(**{**dict(images=64, Ho=28, Wo=28, H=28, W=28, C=128, KH=3, KW=3, N=128, PH=1, PW=1), **k})
    assert K.wgrad_plan(layer()).tile == '128x128'
    assert K.wgrad_plan(layer(C=64, N=64)).tile is not None
    assert K.wgrad_plan(layer(C=125)).tile == '64x64' and K.wgrad_plan(layer(C=3, KH=7, KW=7, PH=3, PW=3)).tile is not None
    assert K.wgrad_plan(layer(N=126)).tile is None and K.wgrad_plan(layer(images=1, C=32)).tile is None
    assert K.wgrad_plan(layer(images=1, H=1, Ho=1, KH=1, PH=0, W=8193, Wo=8193, C=512, N=512)).tile is None
    rows = G(images=1, Ho=200000, Wo=1, H=200000, W=1, C=128, KH=1, KW=1, N=128)
    assert K.wgrad_plan(rows).tile == '128x128'
    for g in (layer(), rows, layer(images=7), layer(C=3, KH=7, KW=7, PH=3, PW=3), layer(C=2048, N=512, KH=1, KW=1, PH=0, PW=0)):
        plan = K.wgrad_plan(g)
        per  = -(-(-(-g.pixels // 32)) // plan.splits)
        assert (plan.splits - 1) * per * 32 < g.pixels <= plan.splits * per * 32          #no slice is empty
    f32 = np.dtype('float32')
    b   = lambda *shape: K.Buffer(None, f32, shape)
    g   = layer(images=2)
    old, new = (K.wgrad_gemm(b(3, g.M * g.N), b(2, 28, 28, 128), b(2, 28, 28, 128), g, 3, tile) for tile in (None, '128x128'))
    assert len(new.params) == len(old.params) + 12 and new.grid == (9 * 1 * 3, 1, 1)


def test_large_kernel_gradients_of_a_program_take_the_kernels():
    x, w, g = np.zeros((16, 28, 28, 64), np.float32), np.zeros((3, 3, 64, 128), np.float32), np.zeros((16, 28, 28, 128), np.float32)
    closed = mj.make_jaxpr(kernel_gradient(padding=P1))(x, w, g)
    kernels = [l.kernel for l in wgrads(JaxprInterpreter(closed, plan_only=True).launches)]
    assert len(kernels) == 1 and kernels[0].startswith('wgrad_split_'), kernels
