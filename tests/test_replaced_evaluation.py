'''What a program puts in front of an evaluation - of the interpreter's or of its sequence's - is gone through by every call, native plan
or not. (CPU, on a stand-in for the device)'''
import numpy as np
import pytest

import vkjax_amd
from vkjax_amd import function

from .test_resident_arguments import interpreter


@pytest.mark.parametrize('where', ['interpreter', 'sequence'])
def test_calls_go_through_it(where, monkeypatch):
    interp, native = interpreter(), []
    def plan(args):
        native.append(args)
        return 'native'
    interp.call_plan = lambda *args: plan
    monkeypatch.setattr(function, 'JaxprInterpreter', lambda *args, **kwargs: interp)
    f = vkjax_amd.wrap(lambda w, x: w * x, frontend='minijax')
    args = [np.ones(20, np.float32)] * 2
    f(*args)
    assert len(interp.sequence.computed_with) == 1 and f(*args) == 'native' and len(native) == 1
    target, name = (interp, 'evaluate') if where == 'interpreter' else (interp.sequence, 'eval')
    real, seen = getattr(target, name), []
    def hooked(*a, **kw):
        seen.append(a)
        return real(*a, **kw)
    setattr(target, name, hooked)
    f(*args)
    assert len(seen) == 1 and len(native) == 1 and len(interp.sequence.computed_with) == 2
