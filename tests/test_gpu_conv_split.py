'''The convolution / matrix-product kernels on the bf16 matrix cores (csrc/kernels/conv_split.h): every operand is taken apart
into three bf16 numbers. Integer-valued data make every product and sum exact, so those results have to be equal; on
random data the error against 64-bit sums is bounded by what three parts and fp32 accumulation can lose.'''
import numpy as np
import pytest

import vkjax_amd
from vkjax_amd import kernels as K
from vkjax_amd import minijax as mj
from vkjax_amd.jaxpr_interpreter import JaxprInterpreter

from .common import check_against_oracle

lax, nn, jnp = mj.lax, mj.nn, mj.numpy
DN = ('NHWC', 'HWIO', 'NHWC')
rng = np.random.RandomState(23)


def ints(shape, low=-4, high=5):
    return rng.randint(low, high, size=shape).astype(np.float32)


def conv(stride=(1, 1), padding='SAME', dilation=(1, 1)):
    return lambda x, k: lax.conv_general_dilated(x, k, stride, padding, rhs_dilation=dilation, dimension_numbers=DN)


def split_kernels(fn):
    return [l.kernel for l in list(fn._jaxpr_interpreters.values())[0].launches if l.kernel.startswith('conv_gemm')]


#rows, columns and contractions around the tile edges (128 rows, 64 or 128 columns, k tiles of 32), one and an odd number
#of k tiles, a contraction that ends inside a k tile, kernel taps outside the image, strides, dilation, negative padding's rows
SHAPES = [
    ('1x1, one k tile',                 [1, 11, 12, 32],  [1, 1, 32, 64],   conv()),
    ('1x1, 127 rows, 3 k tiles',        [1, 127, 1, 96],  [1, 1, 96, 63],   conv()),
    ('1x1, 129 rows, 65 columns',       [1, 129, 1, 64],  [1, 1, 64, 65],   conv()),
    ('1x1, k ends in a tile, 2 rows',   [1, 2, 1, 132],   [1, 1, 132, 130], conv()),
    ('1x1, 4 features',                 [1, 40, 7, 4],    [1, 1, 4, 33],    conv()),
    ('1x1 stride 2',                    [3, 15, 14, 64],  [1, 1, 64, 40],   conv((2, 2))),
    ('3x3 SAME',                        [2, 9, 11, 64],   [3, 3, 64, 70],   conv()),
    ('3x3 VALID, odd number of k tiles', [2, 13, 12, 32], [3, 3, 32, 128],  conv(padding='VALID')),
    ('3x3 stride 2, 96 features',       [2, 15, 15, 96],  [3, 3, 96, 129],  conv((2, 2))),
    ('3x3 dilated',                     [1, 17, 13, 32],  [3, 3, 32, 20],   conv(dilation=(2, 3))),
    ('5x5 SAME',                        [1, 10, 9, 32],   [5, 5, 32, 17],   conv()),
]


@pytest.mark.gpu
@pytest.mark.parametrize('tile', list(K.CONV_SPLIT_TILES))
@pytest.mark.parametrize('desc,xs,ks,f', SHAPES, ids=[s[0] for s in SHAPES])
def test_tile_edges_and_slices(tile, desc, xs, ks, f):
    x, k = ints(xs), ints(ks, -3, 4)
    ktiles = 2 * -(-int(np.prod(ks[:3])) // 64)
    for slices in (1, 2, 3, 7):
        if slices > 1 and ktiles < 2 * slices:
            continue
        print(f'case: {desc}, tile {tile}, {slices} slices', flush=True)
        with K.overrides(conv_split=tile, conv_split_slices=slices):
            _, _, fn = check_against_oracle(f, [x, k], exact=True)
        assert split_kernels(fn) == [f'conv_gemm_split_{tile}'], split_kernels(fn)
        #a second and third evaluation find the counters of the slices at zero again
        first = fn(x, k)
        assert np.array_equal(first, fn(x, k))


@pytest.mark.gpu
@pytest.mark.parametrize('slices', (1, 3))
def test_epilogues_and_second_results(slices):
    '''Batch norm, residual and ReLU in the launch, a centred result stored beside it, and an epilogue in another order.'''
    x, k, r = ints([2, 14, 13, 64]), ints([3, 3, 64, 72], -3, 4), ints([2, 14, 13, 72], -50, 50)
    mean, scale, beta = ints([72]), ints([72], 1, 4), ints([72], -9, 9)
    def bn_residual(x, k, mean, scale, beta, r):
        return nn.relu((conv()(x, k) - mean) * scale + beta + r)
    def centred_too(x, k, mean, scale, beta, r):
        c = conv()(x, k) - mean
        return nn.relu(c * scale + beta), c
    def other_order(x, k, mean, scale, beta, r):
        return (conv()(x, k) * scale - mean) * beta
    for f in (bn_residual, centred_too, other_order):
        with K.overrides(conv_split=True, conv_split_slices=slices):
            _, _, fn = check_against_oracle(f, [x, k, mean, scale, beta, r], exact=True)
        assert len(split_kernels(fn)) == 1 and split_kernels(fn)[0].startswith('conv_gemm_split_')


#epilogues other than (- vector, * vector, + vector, + full tensor, max with a scalar) in this order
STEPS = {'relu6': lambda y, r, v: jnp.minimum(nn.relu(y), 6.0), 'scalar': lambda y, r, v: 0.5 - (y + 2.0) * 0.25, 'quotient': lambda y, r, v: y / v,
         'reciprocal': lambda y, r, v: v / (y * y + 1.0), 'bias, scale': lambda y, r, v: (y + v) * v, 'behind the relu': lambda y, r, v: nn.relu(y) + r,
         'residual, bias': lambda y, r, v: y + r + v, 'difference': lambda y, r, v: y - r, 'difference, left': lambda y, r, v: r - y,
         'two residuals': lambda y, r, v: jnp.maximum((y + r) * r, v - r), 'six steps': lambda y, r, v: (((y + v) * v - r) * 0.5 + r) * v}


@pytest.mark.gpu
@pytest.mark.parametrize('tile', list(K.CONV_SPLIT_TILES))
@pytest.mark.parametrize('name', list(STEPS))
def test_other_epilogues(name, tile):
    x, k, r = ints([2, 14, 13, 64]), ints([3, 3, 64, 72], -3, 4), ints([2, 14, 13, 72], -50, 50)
    v = 2.0 ** ints([72], -2, 3)
    for slices in (1, 3):
        print(f'case: {name}, tile {tile}, {slices} slices', flush=True)
        with K.overrides(conv_split=tile, conv_split_slices=slices):
            #(a quotient by more than a power of two is rounded, by both sides to the nearest)
            check_against_oracle(lambda x, k, r, v: STEPS[name](conv()(x, k), r, v), [x, k, r, v], exact=True)


@pytest.mark.parametrize('name', list(STEPS))
def test_other_epilogues_are_part_of_the_product(name):
    '''Plan only: as behind the fp32 kernels, no launch besides the product and the packing for those that are one chain behind it.'''
    args = [np.zeros(s, np.float32) for s in ((8, 28, 28, 128), (1, 1, 128, 512), (8, 28, 28, 512), (512,))]
    f = lambda x, k, r, v: STEPS[name](conv()(x, k), r, v)
    def launches(choice):
        with K.overrides(conv_split=choice):
            return [l.kernel for l in JaxprInterpreter(mj.make_jaxpr(f)(*args), plan_only=True).launches]
    here, fp32 = launches(True), launches(False)
    assert any(k.startswith('conv_gemm_split') for k in here) and len(here) == len(fp32) + 1, (here, fp32)


LAYOUTS = ('NCHW', 'HWNC', 'CHWN', 'NHWC')


def conv_laid_out(layout):
    return lambda x, k: lax.conv_general_dilated(x, k, (1, 1), 'SAME', dimension_numbers=('NHWC', 'HWIO', layout))


def laid_out(layout):
    per_feature = [72 if d == 'C' else 1 for d in layout]
    return lambda x, k, r, v: nn.relu((conv_laid_out(layout)(x, k) - v.reshape(per_feature)) + r)


@pytest.mark.gpu
@pytest.mark.parametrize('tile', list(K.CONV_SPLIT_TILES))
@pytest.mark.parametrize('layout', LAYOUTS)
def test_results_in_other_layouts(layout, tile):
    size = dict(N=3, H=9, W=11, C=72)
    args = [ints([3, 9, 11, 32]), ints([3, 3, 32, 72], -3, 4), ints([size[d] for d in layout], -50, 50), ints([72])]
    for slices in (1, 3):
        print(f'case: {layout}, tile {tile}, {slices} slices', flush=True)
        with K.overrides(conv_split=tile, conv_split_slices=slices):
            _, _, fn = check_against_oracle(laid_out(layout), args, exact=True)
        assert len(split_kernels(fn)) == 1 and split_kernels(fn)[0].startswith('conv_gemm_split')
        #the backward pass of a ReLU: a second result, both laid out like the activation
        def masked(x, k, r, v):
            m = jnp.where(r > 0, conv_laid_out(layout)(x, k), 0.0)
            return m, m * v.reshape([72 if d == 'C' else 1 for d in layout])
        with K.overrides(conv_split=tile, conv_split_slices=slices):
            check_against_oracle(masked, args, exact=True)


@pytest.mark.parametrize('layout', LAYOUTS)
def test_epilogues_join_products_of_every_layout(layout):
    '''Plan only: the same launches behind the product as with the fp32 kernels.'''
    size = dict(N=8, H=28, W=28, C=72)
    args = [np.zeros(s, np.float32) for s in ([8, 28, 28, 256], [3, 3, 256, 72], [size[d] for d in layout], [72])]
    def launches(choice):
        with K.overrides(conv_split=choice):
            return [l.kernel for l in JaxprInterpreter(mj.make_jaxpr(laid_out(layout))(*args), plan_only=True).launches]
    here, fp32 = launches(True), launches(False)
    assert any(k.startswith('conv_gemm_split') for k in here) and len(here) == len(fp32) + 1, (here, fp32)


@pytest.mark.gpu
def test_gradients_pack_transposed_and_reversed_kernels():
    '''Input gradients of strided and unit-stride convolutions: the kernel operand is packed straight from the forward
    kernel (swapped features, reversed taps, every other tap), results go to every other position of the array.'''
    for stride, xs, ks in (((1, 1), [2, 10, 9, 32], [3, 3, 32, 64]), ((2, 2), [2, 12, 11, 32], [3, 3, 32, 64]), ((2, 2), [1, 9, 9, 64], [1, 1, 64, 32])):
        g = lambda x, k: mj.grad(lambda v, w: (lax.conv_general_dilated(v, w, stride, 'SAME', dimension_numbers=DN) ** 2).sum())(x, k)
        print(f'case: gradient, stride {stride}, {xs} {ks}', flush=True)
        with K.overrides(conv_split=True):
            _, _, fn = check_against_oracle(g, [ints(xs, -2, 3), ints(ks, -2, 3)], exact=True)
        assert sum(name.startswith('conv_gemm_split') for name in split_kernels(fn)) >= 2


@pytest.mark.gpu
@pytest.mark.parametrize('k', (32, 1000, 4608))
def test_error_against_64_bit_sums(k):
    '''|error| <= (2^-24 for the parts left out + (6 k / 16 + 16) 2^-24 for the roundings of the accumulator) sum |x||w|, and not
    above that of the fp32 kernels in the 2-norm (0.4 to 0.9 times measured on data of one scale).'''
    x, w = rng.standard_normal((300, k)).astype(np.float32), rng.standard_normal((k, 96)).astype(np.float32)
    x[:, 0] *= 1e4                                       #parts of very different size in one sum
    exact  = x.astype(np.float64) @ w.astype(np.float64)
    limit  = (6 * k / 16 + 17) * 2.0 ** -24 * (np.abs(x).astype(np.float64) @ np.abs(w).astype(np.float64))
    errors = {}
    for choice in (True, False):
        with K.overrides(conv_split=choice):
            fn = vkjax_amd.wrap(lambda x, w: jnp.dot(x, w), frontend='minijax')
            errors[choice] = np.abs(fn(x, w).astype(np.float64) - exact)
        assert split_kernels(fn)[0].startswith('conv_gemm_split') == choice
    assert (errors[True] <= limit).all()
    assert np.linalg.norm(errors[True]) <= 1.05 * np.linalg.norm(errors[False])


@pytest.mark.gpu
@pytest.mark.parametrize('slices', (1, 2))
def test_infinite_and_huge_operands(slices):
    '''Operands that are infinite, NaN or beyond the largest bf16, in the rows and in the kernel, give what fp32 products give.'''
    x, w = ints([140, 160]), ints([160, 70], -3, 4)
    x[3, 5], x[70, 100], x[139, 159], x[20, 7] = np.inf, -np.inf, np.nan, 3.4e38
    w[9, 2], w[159, 69], w[40, 33], w[41, 33] = np.inf, 3.4e38, -3.4e38, 1.0
    x[:, 159] = np.where(np.isfinite(x[:, 159]), np.sign(x[:, 159]), x[:, 159])
    x[:, 40] = np.sign(x[:, 40])
    results = []
    for choice in (True, False):
        with K.overrides(conv_split=choice, conv_split_slices=slices if choice else None):
            results.append(vkjax_amd.wrap(lambda x, w: jnp.dot(x, w), frontend='minijax')(x, w))
    assert np.array_equal(results[0], results[1], equal_nan=True)
    assert np.isnan(results[0]).any() and np.isinf(results[0]).any() and np.isfinite(results[0]).any()


@pytest.mark.gpu
@pytest.mark.parametrize('tile', list(K.CONV_SPLIT_TILES))
@pytest.mark.parametrize('desc,xs,ks,f', SHAPES, ids=[s[0] for s in SHAPES])
def test_sums_computed_again_with_fp32_products(tile, desc, xs, ks, f):
    '''Over the same shapes, with operands that are not finite (and one beyond the largest bf16) in images and kernel: the sums they reach are
    computed again by another loop over the operands.'''
    x, k = ints(xs), ints(ks, -3, 4)
    k[:, :, -1] = np.sign(k[:, :, -1])                   #(a product beyond the largest number would be infinite or not by the order of its sum)
    x.reshape(-1)[rng.permutation(x.size)[:3]] = np.inf, np.nan, -np.inf
    k.reshape(-1)[rng.permutation(k.size)[:2]] = np.inf, -np.inf
    x[-1, -1, -1, -1] = 3.4e38
    results = []
    print(f'case: {desc}, tile {tile}', flush=True)
    for choice in (tile, False):
        with K.overrides(conv_split=choice):
            results.append(vkjax_amd.wrap(f, frontend='minijax')(x, k))
    assert np.array_equal(results[0], results[1], equal_nan=True) and not np.isfinite(results[0]).all()


def test_plans_and_packed_layout():
    '''Plan only: which products take these kernels, the argument block's tail, and the size of the packed operand.'''
    def plan(m, k, n):
        closed = mj.make_jaxpr(lambda x, w: jnp.dot(x, w))(np.zeros((m, k), np.float32), np.zeros((k, n), np.float32))
        return JaxprInterpreter(closed, plan_only=True)
    interp = plan(12544, 2304, 256)
    assert [l.kernel for l in interp.launches][0] == 'conv_split_pack' and interp.launches[1].kernel.startswith('conv_gemm_split_')
    pack, product = interp.launches
    assert pack.buffers[0][0] is product.buffers[2][0] and pack.buffers[0][0].size * 4 == 8 * 36 * 12288 and pack.grid[0] == 8 * 72 * 2 // 4
    whole, _, slices, each, extra = np.frombuffer(product.params, np.int32)[-5 - 9:-9]
    assert each * slices + extra == 36 and product.grid[0] >= whole
    for m, k, n in ((2048, 4608, 512), (12544, 64, 256), (4096, 256, 32)):          #too few rows, too short a contraction, too little work
        assert all('split' not in l.kernel for l in plan(m, k, n).launches), (m, k, n)


@pytest.mark.parametrize('m,k,n,bf16', [
    (65536, 1024, 32, False), (16384, 4096, 32, False), (50176, 4096, 20, False), (200704, 512, 32, False), (65536, 1024, 33, True),  #columns
    (20000, 2048, 32, True), (32768, 2048, 32, True), (32800, 2048, 32, False), (20000, 1024, 32, False),                             #... up to 1024 tiles of 32 rows
    (4096, 1024, 128, False), (8192, 2048, 64, False), (3136, 3072, 128, False), (4096, 4096, 64, True), (8224, 2048, 64, True),      #few tiles
    (200704, 128, 64, False), (200704, 192, 64, True), (200704, 128, 68, True),                                                        #short and narrow
    (3136, 1024, 256, True), (12544, 512, 128, True), (12544, 64, 1024, False)])                                                       #layers of a network
def test_products_that_the_fp32_kernels_compute_faster_stay_with_them(m, k, n, bf16):
    '''Plan only: sizes that were measured on both sides of every line of the rule, and those beside the lines.'''
    program = JaxprInterpreter(mj.make_jaxpr(jnp.dot)(np.broadcast_to(np.float32(0), (m, k)), np.broadcast_to(np.float32(0), (k, n))), plan_only=True)
    assert any('split' in l.kernel for l in program.launches) == bf16, [l.kernel for l in program.launches]


#input gradients of a strided 1x1 convolution whose result has one position: they write one element in four (or two) of the features'
#array and zeros come from another launch, so what follows cannot be computed with the product
ONE_POSITION = [(130, 2, 2, 64), (129, 1, 2, 64), (131, 2, 1, 64)]
BEHIND = {'relu': lambda d, r, k: nn.relu(d), 'add': lambda d, r, k: d + r, 'scale': lambda d, r, k: d * k,
          'relu backward': lambda d, r, k: jnp.where(r > 0, d, 0.0) * k}


def gradient_of_one_position(behind):
    loss = lambda x, w, ct: (lax.conv_general_dilated(x, w, (2, 2), 'VALID', dimension_numbers=DN) * ct).sum()
    return lambda x, w, ct, r, k: behind(mj.grad(loss)(x, w, ct), r, k)


@pytest.mark.parametrize('behind', list(BEHIND))
@pytest.mark.parametrize('xs', ONE_POSITION)
def test_a_product_that_writes_part_of_its_result_is_not_joined(xs, behind):
    '''Plan only: the result of the program is written by a launch of its own, over all its elements.'''
    args = [np.zeros(s, np.float32) for s in (xs, (1, 1, 64, 96), (xs[0], 1, 1, 96), xs, (64,))]
    with K.overrides(conv_split=True):
        program = JaxprInterpreter(mj.make_jaxpr(gradient_of_one_position(BEHIND[behind]))(*args), plan_only=True)
    out = program.output_buffers[0]
    writers = [l for l in program.launches if any(l.buffers[i][0] is out for i in l.written)]
    assert len(writers) == 1 and writers[0].kernel.startswith('ew_chain'), [l.kernel for l in program.launches]
    assert sum(l.kernel.startswith('conv_gemm_split') for l in program.launches) == 1


@pytest.mark.gpu
@pytest.mark.parametrize('behind', list(BEHIND))
@pytest.mark.parametrize('xs', ONE_POSITION)
def test_values_behind_a_product_that_writes_part_of_its_result(xs, behind):
    args = [ints(xs), ints((1, 1, 64, 96), -3, 4), ints((xs[0], 1, 1, 96)), ints(xs, -9, 10), ints((64,), 1, 4)]
    print(f'case: {xs}, {behind}', flush=True)
    with K.overrides(conv_split=True):
        _, _, fn = check_against_oracle(gradient_of_one_position(BEHIND[behind]), args, exact=True)
    assert len(split_kernels(fn)) == 1 and split_kernels(fn)[0].startswith('conv_gemm_split')
