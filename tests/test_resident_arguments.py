'''What stays in HBM between calls: an evaluation computes with the arguments of its own call, whatever was held there before
(CPU: the evaluation is a stand-in that keeps what it is handed; on the GPU, the results).'''
import ctypes as C
import weakref

import numpy as np
import pytest

import vkjax_amd
from vkjax_amd import hip, minijax as mj
from vkjax_amd.jaxpr_interpreter import JaxprInterpreter


def frozen(x):
    x = x.copy()
    x.flags.writeable = False
    return x


class Sequence:
    '''Keeps what is uploaded, slot by slot, and notes what every evaluation computes with.'''
    def __init__(self, n_inputs):
        self.n_slots, self.hbm, self.computed_with = n_inputs + 1, [None] * n_inputs, []

    def eval(self, host, flags, next_host_arrays=None):
        for these, last in ((host, False), (next_host_arrays or [None] * self.n_slots, True)):
            for slot in range(len(self.hbm)):
                if these[slot] is not None:
                    self.hbm[slot] = these[slot].copy()
            if not last:
                self.computed_with.append([float(x[0]) if x is not None else None for x in (np.asarray(h).view(np.float32) for h in self.hbm)])


def interpreter(**kwargs):
    '''The program w * x on two arrays of 20, on the stand-in.'''
    args = [np.zeros(20, np.float32)] * 2
    interp = JaxprInterpreter(mj.make_jaxpr(lambda w, x: w * x)(*args), plan_only=True, **kwargs)
    interp.sequence, interp._input_slots, interp._input_specs = Sequence(2), [0, 1], [(20, np.dtype(np.float32))] * 2
    interp._output_slots, interp._output_sizes = [2], [20]
    return interp


def full(value, kind=np.copy):
    return kind(np.full(20, value, np.float32))


X = full(0)


@pytest.mark.parametrize('resident', [(), (0,)])
def test_an_array_held_before_another_took_its_place(resident):
    interp = interpreter(resident_argnums=resident)
    a, b = full(1, frozen), full(2)
    for w in (a, a, b, a, b, b, a, full(3, frozen), a):
        interp.run(w, X)
        assert interp.sequence.computed_with[-1][0] == w[0]


def test_one_array_made_writeable_changed_and_made_read_only_again():
    interp = interpreter()
    a = full(1, frozen)
    for value in (1, 3, 5):
        interp.run(a, X)
        assert interp.sequence.computed_with[-1][0] == value
        a.flags.writeable = True
        a += 1
        interp.run(a, X)
        assert interp.sequence.computed_with[-1][0] == value + 1
        a += 1
        a.flags.writeable = False


def test_streams():
    interp = interpreter()
    a, b = full(1, frozen), full(2)
    order = [a, b, a, a, b, b, a]
    for _ in interp.run_stream([(w, X) for w in order]):
        pass
    assert [w[0] for w in interp.sequence.computed_with] == [w[0] for w in order]
    #a call in between takes the place of what the stream had sent ahead
    interp, seen = interpreter(), []
    for _ in interp.run_stream([(w, X) for w in order]):
        seen.append(interp.sequence.computed_with[-1][0])
        interp.run(full(5), X)
        interp.run(a, X)
    assert seen == [w[0] for w in order]


def test_uploads_between_calls():
    '''upload_inputs takes the place of held arrays and of what a stream has sent ahead, as a call does.'''
    class Storage:
        size = 20
        def __init__(self, slot):
            self.slot, self.tensor = slot, self
        def upload(self, words):
            interp.sequence.hbm[self.slot] = words.copy()
    interp = interpreter()
    interp.input_buffers = [Storage(0), Storage(1)]
    a, b = full(1, frozen), full(2, frozen)
    interp.run(a, X)
    interp.upload_inputs(b, X)
    interp.run(a, X)
    assert interp.sequence.computed_with[-1][0] == 1
    seen = []
    for _ in interp.run_stream([(a, X), (a, X), (b, X), (a, X)]):
        seen.append(interp.sequence.computed_with[-1][0])
        interp.upload_inputs(full(7), X)
    assert seen == [1, 1, 2, 1]


def test_arguments_whose_evaluation_never_came():
    '''An argument is held only once the evaluation that uploads it has been made.'''
    a, x, wrong = full(1, frozen), full(2, frozen), np.zeros(3, np.float32)
    wrong.flags.writeable = False
    def runs(interp):
        interp.run(a, x)
        return interp.sequence.computed_with[-1]
    interp = interpreter()
    with pytest.raises(TypeError):
        interp.run(a, wrong)
    assert runs(interp) == [1, 2]
    def raises(then):
        yield a, x
        if then is not None:
            yield a, then
        raise KeyError
    for then, error in ((None, KeyError), (wrong, TypeError)):
        interp = interpreter()
        with pytest.raises(error):
            list(interp.run_stream(raises(then)))
        assert runs(interp) == [1, 2]
    #the iterable makes a call of its own
    interp = interpreter()
    def calls():
        for w in (a, full(3, frozen), full(4)):
            yield w, x
            interp.run(full(9), X)
    for _, w in zip(interp.run_stream(calls()), (1, 3, 4)):
        assert interp.sequence.computed_with[-1] == [w, 2]


def test_native_calls():
    '''The same through a call's native plan.'''
    hbm, computed_with = [None, None], []
    def evaluate(sequence, pointers, n, flags):
        for slot in range(2):
            if pointers[slot]:
                hbm[slot] = (C.c_float * 20).from_address(pointers[slot])[0]
        computed_with.append(hbm[0])
        return 0
    class Interpreter:
        def _evaluated(self, status):
            assert status == 0
    callback, resident, leaf = C.CFUNCTYPE(C.c_int, C.c_uint64, C.POINTER(C.c_void_p), C.c_int, C.c_uint32)(evaluate), {}, lambda slot: ('a', (20,), 'f', slot)
    plan = hip.load_call_module().Plan(Interpreter(), resident, C.cast(callback, C.c_void_p).value, 1, 3, 0, [leaf(0), leaf(1)], leaf(2))
    a, b = full(1, frozen), full(2)
    for w in (a, a, b, a, b, b, a, full(3, frozen), a):
        assert plan((w, X)) is not NotImplemented and computed_with[-1] == w[0]
        assert list(resident) == ([] if w is b else [0])
    for value in (3, 5):
        a.flags.writeable = True
        a[:] = value
        plan((a, X))
        a += 1
        a.flags.writeable = False
        plan((a, X))
        assert computed_with[-2:] == [value, value + 1]


def test_arguments_live_until_a_native_call_ends():
    '''The last reference to an array that was held goes inside a call, and what runs then empties the call's own list.'''
    alive, values = [], []
    def evaluate(sequence, pointers, n, flags):
        alive.append(second() is not None)
        values.append((C.c_float * 20).from_address(pointers[1])[19])
        return 0
    class Interpreter:
        def _evaluated(self, status):
            pass
    callback, resident, leaf = C.CFUNCTYPE(C.c_int, C.c_uint64, C.POINTER(C.c_void_p), C.c_int, C.c_uint32)(evaluate), {}, lambda slot: ('a', (20,), 'f', slot)
    plan = hip.load_call_module().Plan(Interpreter(), resident, C.cast(callback, C.c_void_p).value, 1, 3, 0, [('l', [leaf(0), leaf(1)])], leaf(2))
    for kind in (frozen, np.copy):
        old = full(1, frozen)
        arguments = [old, full(3)]
        second = weakref.ref(arguments[1])
        plan((arguments,))
        weakref.finalize(old, lambda: following.clear())
        #the note of `old` gives way to another one, or goes
        following = [full(4, kind), full(5)]
        second = weakref.ref(following[1])
        del old, arguments
        plan((following,))
        assert following == [] and alive[-1] and values[-1] == 5
        assert second() is None


# ------------------------------------------------------------------ on the GPU

@pytest.mark.gpu
def test_a_stream_that_ends_in_an_error():
    f = vkjax_amd.wrap(lambda w, x: w * x, frontend='minijax')
    rng = np.random.default_rng(6)
    a, b = frozen(rng.random(300, dtype=np.float32)), frozen(rng.random(300, dtype=np.float32))
    f(b, b)
    def raises():
        yield a, b
        raise KeyError
    with pytest.raises(KeyError):
        list(f.stream(raises()))
    assert np.array_equal(f(a, b), a * b)


@pytest.mark.gpu
@pytest.mark.parametrize('way', ['plan', 'general', 'stream'])
def test_results_of_calls_in_turn(way):
    f = vkjax_amd.wrap(lambda w, x: w * x + np.float32(1), frontend='minijax')
    rng = np.random.default_rng(5)
    x = rng.random(300, dtype=np.float32)
    a, b, c = frozen(rng.random(300, dtype=np.float32)), rng.random(300, dtype=np.float32), frozen(rng.random(300, dtype=np.float32))
    order = [a, b, a, a, c, b, c, a]
    if way == 'stream':
        results = list(f.stream([(w, x) for w in order]))
    else:
        results = []
        for w in order:
            results.append(f(w, x))
            if way == 'general':
                f._plans = []
    for w, y in zip(order, results):
        assert np.array_equal(y, w * x + np.float32(1))
