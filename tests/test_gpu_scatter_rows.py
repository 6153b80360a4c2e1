'''Sorted scatter-adds: more slots per row than a wave has lanes, and several short rows per wave. The sums have the bits of a sequential loop.'''
import numpy as np
import pytest

import vkjax_amd
from vkjax_amd import kernels as K, minijax as mj
from vkjax_amd.jaxpr_interpreter import JaxprInterpreter

pytestmark = pytest.mark.gpu


def scatter(table, idx, updates):
    return mj.numpy.index_add(table, idx, updates)


def onto_zeros(shape):
    return lambda idx, updates: mj.numpy.index_add(mj.numpy.zeros(shape, np.float32), idx, updates)


def indices(rng, rows, counts, n):
    '''Rows with the given numbers of updates, from the first and from the last one on, some beyond the table and the others anywhere, mixed.'''
    some = np.concatenate([np.full(c, r) for r, c in enumerate(counts)] + [np.full(c, rows - 1 - r) for r, c in enumerate(counts) if rows > 2 * len(counts)])
    rest = rng.integers(0, rows, size=max(0, n - some.size))
    rest[:3] = rows
    return rng.permutation(np.concatenate([some, rest])).astype(np.int32)


def check(rows, cols, idx, dtype, kernel, **choices):
    rng   = np.random.default_rng(rows + cols)
    make  = (lambda *s: rng.standard_normal(s).astype(np.float32)) if dtype == np.float32 else (lambda *s: rng.integers(-99, 99, size=s).astype(dtype))
    table, updates = make(rows, cols), make(idx.size, cols)
    inside = (idx >= 0) & (idx < rows)
    with K.overrides(scatter_sort_threshold=0, **choices):
        fn = vkjax_amd.wrap(scatter, frontend='minijax')
        for t, i, u in ((table, idx, updates), (table, idx[::-1].copy(), updates[::-1].copy())):
            want = t.copy()
            keep = inside if i is idx else inside[::-1]
            np.add.at(want, i[keep], u[keep])
            assert np.array_equal(fn(t, i, u), want)
        assert list(fn._jaxpr_interpreters.values())[0].launches[-1].kernel == kernel
        if dtype == np.float32:
            want = np.zeros_like(table)
            np.add.at(want, idx[inside], updates[inside])
            assert np.array_equal(vkjax_amd.wrap(onto_zeros(table.shape), frontend='minijax')(idx, updates), want)


#rows that do not fill the last wave, rows of one number up to 32 lanes; buckets of none up to beyond the 16 that are sorted together, up to the slots and beyond
@pytest.mark.parametrize('cols,vec', [(1, 1), (3, 1), (4, 4), (16, 4), (17, 1), (31, 1), (36, 4), (60, 4), (64, 4), (128, 4)])
@pytest.mark.parametrize('dtype', [np.float32, np.int32])
def test_several_rows_per_wave(cols, vec, dtype):
    print('short rows:', cols, dtype.__name__, flush=True)
    rng = np.random.default_rng(cols)
    for rows, cap in ((1, 8), (67, 8), (131, 32), (300, 128)):
        idx = indices(rng, rows, (0, 1, 2, 15, 16, 17, 32, 33, 64, 65, 130, 3, 4, 5)[:rows], 500)
        check(rows, cols, idx, dtype, f'scatter_rows_sum_short_{"f" if dtype == np.float32 else "i"}_v{vec}', scatter_short_rows=True, scatter_bucket_cap=cap)


@pytest.mark.parametrize('cap', (65, 128, 1024))
@pytest.mark.parametrize('cols', (5, 256))
def test_more_slots_than_lanes(cols, cap):
    print('slots:', cols, cap, flush=True)
    idx = indices(np.random.default_rng(cap), 40, (0, 63, 64, 65, 66, 127, 128, 129, 1023, 1024, 1025, 4096, 5), 9000)
    check(40, cols, idx, np.float32, f'scatter_rows_sum_f_v{4 if cols % 4 == 0 else 1}', scatter_short_rows=False, scatter_bucket_cap=cap)


def test_slots_by_the_rule():
    plan = lambda rows, cols, n: [l.kernel for l in JaxprInterpreter(mj.make_jaxpr(scatter)(*[np.zeros(s, t) for s, t in (((rows, cols), np.float32), ((n,), np.int32), ((n, cols), np.float32))]),
                                                                     plan_only=True).launches]
    assert plan(20000, 16, 60000)[-1] == 'scatter_rows_sum_short_f_v4' and plan(20000, 128, 60000)[-1] == 'scatter_rows_sum_f_v4'
    assert plan(20000, 16, 200000)[-1] == 'scatter_rows_sum_f_v4' and plan(2000, 16, 20000)[-1] == 'scatter_rows_sum_f_v4'
    caps = [K.choose_scatter_bucket_cap(n, rows, cols) for n, rows, cols in ((262144, 65536, 256), (32000, 100000, 24), (262144, 1000, 256), (90000, 5000, 200), (1000, 3000000, 16), (5, 2**27, 4))]
    assert caps == [16, 8, 1024, 128, 4, 0]
    assert all(cap * rows <= max(8 * n, 1 << 24) for cap, (n, rows) in zip(caps, ((262144, 65536), (32000, 100000), (262144, 1000), (90000, 5000), (1000, 3000000), (5, 2**27))))


def test_crowded_neighbours_do_not_share_a_wave():
    '''Sixteen rows with a thousand updates each take about as long next to each other as far apart (in one wave, one after the other: some ten times as long).'''
    rows, cols, each = 20000, 16, 1000
    def time(crowded):
        idx = np.repeat(np.asarray(crowded, np.int32), each)
        program = JaxprInterpreter(mj.make_jaxpr(scatter)(*(args := [np.zeros((rows, cols), np.float32), idx, np.ones((idx.size, cols), np.float32)])))
        assert program.launches[-1].kernel == 'scatter_rows_sum_short_f_v4'
        program.upload_inputs(*args)
        best = min(program.replay(2) for _ in range(6))
        y, = program.read_outputs()
        assert (y[crowded] == each).all() and y.sum() == idx.size * cols
        return best
    with K.overrides(scatter_sort_threshold=0):
        apart, neighbours = time([997 * k + 5 for k in range(16)]), time(list(range(4096, 4096 + 16)))
    print('crowded rows apart, neighbours:', apart, neighbours, flush=True)
    assert neighbours < 3 * apart
