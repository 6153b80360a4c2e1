'''Native plans of calls (csrc/call.cpp): which calls they recognise, what they copy, what they hand out - against the general path
(CPU: the evaluation is a stand-in that looks at the pointers), and on the GPU the same results.'''
import ctypes as C
import gc
import sys

import numpy as np
import pytest

import vkjax_amd
from vkjax_amd import hip, minijax as mj, workloads as W

from .common import assert_tree_close

EVAL = C.CFUNCTYPE(C.c_int, C.c_uint64, C.POINTER(C.c_void_p), C.c_int, C.c_uint32)


class Interpreter:
    def __init__(self):
        self.evaluations, self.statuses = 0, []

    def _evaluated(self, status):
        self.evaluations += 1
        self.statuses.append(status)
        if status:
            raise hip.HipError(f'status {status}')


class Harness:
    '''A plan over arguments (dict a: [2, 3] float32, b: int32 scalar, (x: [4] uint32, None)), list [unread [2]]; results (dict of [2, 3] float32, [4] uint32).'''
    def __init__(self):
        self.interpreter, self.resident, self.seen, self.status = Interpreter(), {}, [], 0
        def evaluate(sequence, pointers, n, flags):
            self.seen.append((sequence, [pointers[k] for k in range(n)], flags))
            if not self.status:
                (C.c_float * 6).from_address(pointers[3])[:] = [1, 2, 3, 4, 5, 6]
                (C.c_uint32 * 4).from_address(pointers[4])[:] = [7, 8, 9, 10]
            return self.status
        self.callback = EVAL(evaluate)
        self.arguments = [('d', ['a', 'b'], [('a', (2, 3), 'f', 0), ('a', (), 'i', 1)]), ('t', [('a', (4,), 'u', 2), ('n',)]), ('l', [('a', (2,), 'f', -1)])]
        self.plan = hip.load_call_module().Plan(self.interpreter, self.resident, C.cast(self.callback, C.c_void_p).value, 77, 5, 4, self.arguments,
                                                ('t', [('d', ['y'], [('a', (2, 3), 'f', 3)]), ('a', (4,), 'u', 4)]))

    def args(self):
        return ({'b': np.array(5, np.int32), 'a': np.ones((2, 3), np.float32)}, (np.arange(4, dtype=np.uint32), None), [np.zeros(2, np.float32)])


def frozen(x):
    x = x.copy()
    x.flags.writeable = False
    return x


def test_results_and_pointers():
    h, args = Harness(), Harness().args()
    y = h.plan(args)
    assert type(y) is tuple and list(y[0]) == ['y'] and np.array_equal(y[0]['y'], [[1, 2, 3], [4, 5, 6]]) and np.array_equal(y[1], [7, 8, 9, 10])
    assert y[0]['y'].dtype == np.float32 and y[1].dtype == np.uint32 and y[1].flags.writeable and y[1].flags.owndata
    (sequence, pointers, flags), = h.seen
    assert (sequence, flags) == (77, 4)
    assert pointers[:3] == [args[0]['a'].ctypes.data, args[0]['b'].ctypes.data, args[1][0].ctypes.data] and pointers[3:] == [y[0]['y'].ctypes.data, y[1].ctypes.data]
    assert h.resident == {} and h.interpreter.evaluations == 1


def test_calls_it_does_not_recognise_change_nothing():
    h = Harness()
    class List(list): pass
    class Array(np.ndarray): pass
    a, t, l = h.args()
    others = [(a, t), (a, t, l, l), ({'a': a['a']}, t, l), ({**a, 'c': a['a']}, t, l), ({'a': a['a'], 'c': a['b']}, t, l), (a, list(t), l), (a, t, tuple(l)), (a, t, List(l)),
              (a, (t[0], 0), l), (a, (t[0],), l), ([a['a'], a['b']], t, l), (None, t, l), (a, t, [None]), (a, t, [[1.0, 2.0]]), (a, t, [np.zeros(3, np.float32)]),
              ({**a, 'a': np.ones((3, 2), np.float32)}, t, l), ({**a, 'a': np.ones((2, 3), np.float64)}, t, l), ({**a, 'a': np.ones((2, 3), np.int32)}, t, l),
              ({**a, 'a': np.ones((2, 3), '>f4')}, t, l), ({**a, 'a': np.ones((3, 2), np.float32).T}, t, l), ({**a, 'a': np.ones((2, 6), np.float32)[:, ::2]}, t, l),
              ({**a, 'a': np.ones((2, 3), np.float32).view(Array)}, t, l), ({**a, 'b': 5}, t, l), ({**a, 'b': np.int32(5)}, t, l), ({**a, 'b': np.array([5], np.int32)}, t, l),
              (a, (t[0].astype(np.int32), None), l)]
    for args in others:
        assert h.plan(args) is NotImplemented, args
    assert h.seen == [] and h.resident == {} and h.interpreter.evaluations == 0
    #an unread argument need not be contiguous, keys may come in any order
    assert h.plan((a, t, [np.zeros(4, np.float32)[::2]])) is not NotImplemented and h.plan(({'a': a['a'], 'b': a['b']}, t, l)) is not NotImplemented
    for bad in ((), (1,), ([],), (a, t)):
        with pytest.raises(TypeError):
            h.plan(*bad)


def test_read_only_arrays_are_copied_once():
    h = Harness()
    a, t, l = h.args()
    a = {'a': frozen(a['a']), 'b': a['b']}
    copied = lambda: [p is not None for p in h.seen[-1][1][:3]]
    h.plan((a, t, l)); assert copied() == [True, True, True] and h.resident[0][0] is a['a'] and list(h.resident) == [0]
    h.plan((a, t, l)); assert copied() == [False, True, True]
    a2 = {**a, 'a': frozen(a['a'])}                                            #another object of the same values
    h.plan((a2, t, l)); assert copied() == [True, True, True]
    h.plan((a2, t, l)); assert copied() == [False, True, True]
    view = np.ones((2, 3), np.float32)
    locked = view[:]
    locked.flags.writeable = False                                             #read-only itself, its base is not
    for _ in range(2):
        h.plan(({**a, 'a': locked}, t, l)); assert copied() == [True, True, True]
    data = np.frombuffer(np.ones(6, np.float32).tobytes(), np.float32).reshape(2, 3)
    h.plan(({**a, 'a': data}, t, l)); assert copied() == [True, True, True]
    h.plan(({**a, 'a': data}, t, l)); assert copied() == [False, True, True]
    data2 = frozen(np.ones((2, 3), np.float32))
    h.plan(({**a, 'a': data2}, t, l))
    data2.flags.writeable = True                                               #no longer: copied on every call
    for _ in range(2):
        h.plan(({**a, 'a': data2}, t, l)); assert copied() == [True, True, True]
    h.resident[0] = (a['a'], b'what a check of the memory found')              #noted by the general path for an argument it checks
    h.plan((a, t, l)); assert copied() == [True, True, True]


def test_failed_evaluations_raise_and_references_balance():
    h = Harness()
    args = h.args()
    keep = [sys.getrefcount(x) for x in (args[0]['a'], args[1][0])]
    h.status = 3
    for _ in range(50):
        with pytest.raises(hip.HipError, match='status 3'):
            h.plan(args)
    h.status = 0
    for _ in range(50):
        h.plan(args)
        h.plan((args[0], args[1], []))
    assert h.interpreter.statuses == [3] * 50 + [0] * 50
    gc.collect()
    assert [sys.getrefcount(x) for x in (args[0]['a'], args[1][0])] == keep


def test_specifications_are_checked():
    h = Harness()
    make = lambda arguments, result, slots=5: hip.load_call_module().Plan(h.interpreter, {}, 1, 1, slots, 0, arguments, result)
    leaf = ('a', (2,), 'f', 0)
    for arguments, result in (([('a', (2,), 'f', 5)], leaf), ([leaf], ('a', (2,), 'f', -1)), ([leaf], ('a', (2,), 'f', 7)), ([()], leaf), ([7], leaf),
                              ([('d', ['a'], [])], leaf), ([('a', [2], 'f', 0)], leaf), ([leaf], ())):
        with pytest.raises((TypeError, ValueError)):
            make(arguments, result)


# ------------------------------------------------------------------ on the GPU

@pytest.mark.gpu
def test_calls_equal_the_general_path():
    params, x = W.mlp_inputs(3, 64, (40, 30, 20, 10))
    native, general = (vkjax_amd.wrap(W.mlp, frontend='minijax') for _ in range(2))
    calls = []
    for batch in (64, 7, 64, 1, 7):                                            #several signatures, taken in turn
        for weights in (params, mj.tree_util.tree_map(frozen, params)):
            xs = np.random.default_rng(batch).random((batch, 40), dtype=np.float32)
            general._plans = []
            assert_tree_close(native(weights, xs), general(weights, xs), exact=True, what=f'batch {batch}')
            calls.append(len(native._plans))
    assert calls[-1] == 3
    ro = mj.tree_util.tree_map(frozen, params)
    first = native(ro, x[:64])
    interp = native._get_or_create_jaxpr_interpreter((ro, x[:64]))[0]
    assert len(interp._resident_leaves) == len(mj.tree_util.tree_leaves(ro))
    count = interp._evaluations
    assert_tree_close(native(ro, x[:64]), first, exact=True)
    assert interp._evaluations == count + 1
    #results are the caller's: a later call does not write into them
    kept = [np.copy(l) for l in mj.tree_util.tree_leaves(first)]
    native(ro, -x[:64])
    assert all(np.array_equal(a, b) for a, b in zip(kept, mj.tree_util.tree_leaves(first)))
    #arguments the plans do not take: converted as before
    assert_tree_close(native(ro, np.asfortranarray(x[:64])), first, exact=True)


@pytest.mark.gpu
def test_labels_flags_and_scalars():
    def f(tree, k):
        return {'sum': tree['x'].sum() if hasattr(tree['x'], 'sum') else mj.numpy.sum(tree['x']), 'pair': [tree['x'] * k, mj.numpy.argmax(tree['x'], axis=1)]}, tree['x'] > k
    x = np.random.default_rng(1).standard_normal((5, 6)).astype(np.float32)
    fn = vkjax_amd.wrap(f, frontend='minijax')
    for _ in range(3):
        (first, flags) = fn({'x': x}, np.float32(0.5))
        assert flags.dtype == np.bool_ and np.array_equal(flags, x > 0.5) and np.array_equal(first['pair'][1], x.argmax(axis=1)) and first['sum'].shape == ()
    assert fn._plans == []                                                      #a result of booleans is converted on the host
