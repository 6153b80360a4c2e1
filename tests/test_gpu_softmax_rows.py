'''The softmax launch over the row lengths at which its variants begin and end, and over numbers of rows that leave a wave
or a block partly empty: the bits of the five launches it stands for, and 64-bit values within fp32's reach.'''
import numpy as np
import pytest

import vkjax_amd
from vkjax_amd import minijax as mj, kernels as K

pytestmark = pytest.mark.gpu

#a vector per lane holds 64 resp. 256 values; the last and the first row of neighbouring variants, and odd lengths between them
LENGTHS = [2, 3, 4, 7, 8, 12, 31, 33, 63, 64, 65, 127, 130, 252, 255, 256, 260, 257, 511, 512, 513, 516, 767, 768, 769, 772, 1000, 1023,
           1025, 1028, 1535, 1536, 1537, 1540, 2047, 2049, 2052, 3071, 3072, 3073, 3076, 4091, 4092, 4095]


def test_a_row_fits_its_variant():
    for length in range(1, K.SOFTMAX_MAX_ROW):
        vec = 4 if length % 4 == 0 else 1
        assert any(n * 64 * vec >= length for n in K.SOFTMAX_VECTORS[vec])


@pytest.mark.parametrize('cols', LENGTHS)
def test_softmax_rows(cols):
    rng = np.random.default_rng(cols)
    def f(x):
        p = mj.nn.softmax(x, axis=-1)
        return p, mj.numpy.argmax(p, axis=1)
    for rows in (2, 67):
        x = (rng.standard_normal((rows, cols)) * 4).astype(np.float32)
        x[rows // 2, cols - 1] = np.inf if rows > 2 else 40.0
        if rows > 2:
            x[1, 0], x[2, :], x[3, cols // 2], x[4, cols - 1] = np.nan, -np.inf, -np.inf, 3e38
        print(f'softmax {rows} x {cols}', flush=True)
        fused, unfused = (vkjax_amd.wrap(f, frontend='minijax', fuse=fuse) for fuse in (True, False))
        (p, labels), (q, expected) = fused(x), unfused(x)
        kernels = [l.kernel for l in list(fused._jaxpr_interpreters.values())[0].launches]
        assert len(kernels) == 1 and kernels[0].startswith('softmax_rows'), kernels
        assert np.array_equal(p, q, equal_nan=True) and np.array_equal(labels, expected)
        finite = np.isfinite(x).all(axis=1)
        e = np.exp(x[finite].astype(np.float64) - x[finite].max(axis=1, keepdims=True))
        #x - max is rounded to fp32: up to 2^-24 of 1e2 in the exponent for these rows (3e38: the others vanish), then a few ulp
        assert np.allclose(p[finite], e / e.sum(axis=1, keepdims=True), rtol=1e-5, atol=1e-37)
