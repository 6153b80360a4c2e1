'''Uploads of parts of arrays (vkj_seq_record_upload with an offset and a size) change those parts and nothing else, and of two that
overlap the one recorded last stays: on the CPU build of the runtime, with and without the kernel that carries small ranges
(whose stand-in takes the ranges in another order than they were given in).'''
import ctypes as C

import numpy as np
import pytest

from vkjax_amd import hip

from .test_shim_cpu import H, World, lib     # noqa: F401 (the fixture)


@pytest.fixture(params=[False, True], ids=['transfers', 'carried'])
def world(lib, request):                     # noqa: F811
    lib.fake_hip_carry(int(request.param))
    w = World(lib)
    yield w
    lib.fake_hip_carry(0)
    w.close()


#arrays of these sizes (packed together below 64 KB), the uploads (array, first byte, bytes) and whether 8 MB of another array, from which on
#arguments are sent as one stream of chunks, come with them
CASES = {
    'two parts of one':        ([256], [(0, 0, 4), (0, 64, 4)]),
    'parts that meet':         ([256], [(0, 0, 64), (0, 64, 32)]),
    'a whole one and a part':  ([200, 300], [(0, 0, 200), (1, 64, 100)]),
    'a part and a whole one':  ([200, 300], [(0, 0, 100), (1, 0, 300)]),
    'whole ones':              ([200, 4, 256, 300], [(0, 0, 200), (1, 0, 4), (2, 0, 256), (3, 0, 300)]),
    'odd bytes':               ([300], [(0, 0, 4), (0, 33, 5), (0, 41, 4)]),
    'one inside another':      ([300], [(0, 0, 300), (0, 100, 8)]),
    'one around another':      ([300], [(0, 100, 8), (0, 0, 300)]),
    'two in their middle':     ([300], [(0, 0, 200), (0, 100, 200)]),
    'inside, unpacked':        ([100000], [(0, 0, 100000), (0, 4096, 8)]),
    'around, unpacked':        ([100000], [(0, 4096, 8), (0, 0, 100000)]),
    'odd inside, unpacked':    ([100000], [(0, 0, 100000), (0, 4097, 2)]),
    'many':                    ([100000], [(0, 4 * k, 400) for k in range(0, 1000, 25)]),
    'inside, large':           ([9 << 20], [(0, 0, 9 << 20), (0, 5 << 20, 8)]),
}


@pytest.mark.parametrize('large', [False, True])
@pytest.mark.parametrize('case', CASES)
def test_parts(world, case, large):
    lib, rng = world.lib, np.random.default_rng(3)
    sizes, uploads = CASES[case]
    sizes, uploads = list(sizes), list(uploads)
    if large:
        uploads.append((len(sizes), 0, 9 << 20))
        sizes.append(9 << 20)
    bufs, expected = [], []
    for n in sizes:
        b = H()
        alloc = lib.vkj_buf_alloc_packed if n <= 65536 else lib.vkj_buf_alloc
        assert alloc(world.ctx, n, C.byref(b)) == 0
        bufs.append(b)
        expected.append(rng.integers(0, 256, n, dtype=np.uint8))
        assert lib.vkj_buf_upload(world.ctx, b, 0, expected[-1].ctypes.data, n) == 0
    seq = H()
    assert lib.vkj_seq_create(world.ctx, 0, C.byref(seq)) == 0
    for slot, (k, at, n) in enumerate(uploads):
        assert lib.vkj_seq_record_upload(seq, bufs[k], at, slot, n) == 0
    for _ in range(2):
        host = [rng.integers(0, 256, n, dtype=np.uint8) for _, _, n in uploads]
        for (k, at, n), h in zip(uploads, host):
            expected[k][at:at + n] = h
        pointers = (C.c_void_p * len(host))(*[h.ctypes.data for h in host])
        assert lib.vkj_seq_eval(seq, pointers, len(host), 0) == 0, lib.vkj_last_error()
        for k, n in enumerate(sizes):
            got = np.empty(n, np.uint8)
            assert lib.vkj_buf_download(world.ctx, bufs[k], 0, got.ctypes.data, n) == 0
            assert np.array_equal(got, expected[k]), (k, np.flatnonzero(got != expected[k])[:8])
    #one of them alone
    pointers = (C.c_void_p * len(host))(host[0].ctypes.data)
    assert lib.vkj_seq_eval(seq, pointers, len(host), hip.EVAL_NULL_IS_RESIDENT) == 0
    k, at, n = uploads[0]
    expected[k][at:at + n] = host[0]
    got = np.empty(sizes[k], np.uint8)
    assert lib.vkj_buf_download(world.ctx, bufs[k], 0, got.ctypes.data, sizes[k]) == 0
    assert np.array_equal(got, expected[k])
    assert lib.vkj_seq_destroy(seq) == 0
    for b in bufs:
        assert lib.vkj_buf_free(world.ctx, b) == 0
