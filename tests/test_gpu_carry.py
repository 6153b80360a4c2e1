'''Small arguments and results are carried between pinned host memory and HBM by a kernel (carry_ranges in csrc/static_landing.hip): sizes around its
vectors and blocks, runs of packed neighbours with gaps between them, more ranges than one table holds, resident neighbours that stay as they are.'''
import numpy as np
import pytest

import vkjax_amd
from vkjax_amd import minijax as mj

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('sizes', [(1,), (3, 4, 5), (63, 64, 65, 1), (1023, 1024, 1025), (16384, 16385, 7), (40000, 1, 65536, 65537, 2), (1 << 20, (1 << 20) - 1),
                                   tuple(range(1, 41)), (20000,) * 20], ids=lambda s: f'{len(s)} of {max(s)}')
def test_arguments_and_results_arrive(sizes):
    rng = np.random.default_rng(len(sizes) + sizes[0])
    f   = lambda *xs: [x + np.float32(1) for x in xs] + [xs[0] * xs[0], mj.numpy.sum(xs[-1])]
    fn  = vkjax_amd.wrap(f, frontend='minijax')
    for call in range(4):
        xs = [rng.integers(-99, 99, n).astype(np.float32) for n in sizes]
        ys = fn(*xs)
        for x, y in zip(xs, ys):
            assert np.array_equal(y, x + 1), (call, x.size)
        assert np.array_equal(ys[-2], xs[0] ** 2)


def test_resident_neighbours_keep_their_values():
    '''Every other one of a row of small arguments is read-only and stays in HBM: what is carried past it leaves it alone.'''
    rng = np.random.default_rng(5)
    f   = lambda *xs: [x * np.float32(2) for x in xs]
    fn  = vkjax_amd.wrap(f, frontend='minijax')
    fixed = [rng.integers(-99, 99, n).astype(np.float32) for n in (1, 60, 64, 65, 127, 128, 3)]
    for x in fixed:
        x.flags.writeable = False
    for call in range(4):
        xs = [v for x in fixed for v in (x, rng.integers(-99, 99, 64 + call).astype(np.float32))]
        for which in (xs, xs[:-1] + [np.zeros_like(xs[-1])]):
            for x, y in zip(which, fn(*which)):
                assert np.array_equal(y, 2 * x)
