'''Draws of an odd number of words as one launch: the counters padded with one zero, the last word dropped (fusion.fuse_random_streams).'''
import numpy as np
import pytest

import vkjax_amd
from vkjax_amd import minijax as mj
from vkjax_amd.jaxpr_interpreter import JaxprInterpreter

jnp, lax, r = mj.numpy, mj.lax, mj.random
KEY = r.PRNGKey(23)


def kernels(f, *args):
    return [l.kernel for l in JaxprInterpreter(mj.make_jaxpr(f)(*args), plan_only=True).launches]


#one vector per thread and several, h a multiple of 4 and not, one word in the last workgroup
@pytest.mark.gpu
@pytest.mark.parametrize('shape', ((1,), (3,), (5, 1), (7,), (11, 13), (511,), (513,), (4097,), (1001, 1001), (3, (1 << 20) + 1)))
def test_bits_are_those_of_the_separate_launches(shape):
    def uniform(key):
        return r.uniform(r.split(key)[1], shape)
    def interval(key):
        return r.uniform(key, shape, minval=-2.0, maxval=3.0)
    def bits(key):
        return r.random_bits(key, shape)
    def normal(key):
        return r.normal(key, shape)
    for f in (uniform, interval, bits, normal):
        print(f'{f.__name__} {shape}', flush=True)
        a, b = (np.asarray(vkjax_amd.wrap(f, frontend='minijax', fuse=fuse)(KEY)) for fuse in (True, False))
        assert np.array_equal(a, b), f.__name__


def test_what_becomes_one_launch():
    '''Plan only. Counters that are padded with anything but a zero, or read elsewhere too, stay as they are.'''
    assert kernels(lambda key: r.uniform(r.split(key)[1], (11, 13)), KEY) == ['threefry2x32_stream_v1_uniform']
    assert kernels(lambda key: r.random_bits(key, (4097,)), KEY) == ['threefry2x32_stream_v1']

    def by_hand(pad, both=False, front=False):
        def f(key):
            k    = [lax.reshape(lax.slice(key, (i,), (i + 1,)), ()) for i in (0, 1)]
            ends = [lax.iota(np.uint32, 255), pad]
            c    = jnp.concatenate(ends[::-1] if front else ends)
            y    = lax.threefry2x32(*k, lax.slice(c, (0,), (128,)), lax.slice(c, (128,), (256,)))
            out  = lax.slice(jnp.concatenate(y), (0,), (255,))
            return (out, c) if both else out
        return kernels(f, KEY)
    zero, one = np.zeros((1,), np.uint32), np.ones((1,), np.uint32)
    assert by_hand(zero) == ['threefry2x32_stream_v1']
    for stays in (by_hand(one), by_hand(zero, both=True), by_hand(zero, front=True)):
        assert any(k.startswith('threefry2x32_k') for k in stays), stays
