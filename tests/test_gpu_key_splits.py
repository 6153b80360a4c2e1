'''Draws whose kernel computes the split of its key itself (threefry_split_word in csrc/kernels/threefry.hip).'''
import numpy as np
import pytest

import vkjax_amd
from vkjax_amd import minijax as mj, ops


@pytest.mark.gpu
@pytest.mark.parametrize('layout', ('traced', 'halves', 'partitionable'))
@pytest.mark.parametrize('size', (1, 2, 6, 8, 255, 1024, 4096 * 8, (1 << 21) + 8, 3 << 21))
def test_draws_that_split_their_key_themselves(size, layout, monkeypatch):
    '''A draw behind a key split is one launch: the same bits as the separate ones, for sizes of one and of several vectors per thread, keys at both
    ends of splits of even and odd numbers, splits of splits, and splits that something else reads too (which stay).'''
    r = mj.random
    monkeypatch.setattr(ops, 'THREEFRY_PARTITIONABLE', layout == 'partitionable')
    previous = r.key_primitives(layout != 'traced')
    try:
        check(r, size, 0 if layout == 'traced' else 1)
    finally:
        r.key_primitives(previous)


def check(r, size, copies):
    '''`copies`: launches that copy a key out of a split which stays.'''
    def last_of_two(key):
        return r.uniform(r.split(key)[1], (size,))
    def of_seven(key):
        keys = r.split(key, 7)
        return r.uniform(keys[0], (size,)), r.random_bits(keys[6], (size,)), r.uniform(keys[3], (size,), minval=-2.0, maxval=3.0)
    def nested(key):
        return r.uniform(r.split(r.split(key, 3)[2])[0], (size,))
    def shared(key):
        keys = r.split(key)
        return r.uniform(keys[1], (size,)), keys
    key = r.PRNGKey(17)
    for f, launches in ((last_of_two, 1), (of_seven, 3), (nested, 2 + copies), (shared, 2 + copies)):
        print(f'{f.__name__} {size}', flush=True)
        fused, unfused = (vkjax_amd.wrap(f, frontend='minijax', fuse=fuse) for fuse in (True, False))
        for a, b in zip(mj.tree_util.tree_leaves(fused(key)), mj.tree_util.tree_leaves(unfused(key))):
            assert np.array_equal(a, b), (f.__name__, size)
        kernels = [l.kernel for l in list(fused._jaxpr_interpreters.values())[0].launches]
        assert size % 2 or len(kernels) == launches, (f.__name__, kernels)
