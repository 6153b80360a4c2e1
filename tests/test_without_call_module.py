'''A package whose extension module of native calls has not been built (or does not fit this Python) still runs: calls take the
general path. (CPU)'''
import warnings

import numpy as np
import pytest

from vkjax_amd import hip, minijax as mj
from vkjax_amd.csrc import build
from vkjax_amd.jaxpr_interpreter import JaxprInterpreter
from vkjax_amd.minijax import tree_util


@pytest.mark.parametrize('content', [None, b'no shared object'])
def test_calls_take_the_general_path(tmp_path, monkeypatch, content):
    monkeypatch.setattr(hip, 'LIBDIR', str(tmp_path))
    monkeypatch.setattr(hip, '_call_module', None)
    if content is not None:
        (tmp_path / 'vkjax_call.so').write_bytes(content)
    args   = [np.zeros(20, np.float32)] * 2
    interp = JaxprInterpreter(mj.make_jaxpr(lambda w, x: w * x)(*args), plan_only=True)
    class Sequence:
        handle, n_slots = 1, 3
    interp.sequence, interp._input_slots, interp._output_slots = Sequence(), [0, 1], [2]
    plan = lambda: interp.call_plan(args, tree_util.tree_flatten(args)[1].children, tree_util.tree_structure(args[0]))
    with pytest.warns(RuntimeWarning, match='vkjax_call'):
        assert plan() is None
    with warnings.catch_warnings():
        warnings.simplefilter('error')                          #said once
        assert plan() is None
    with pytest.raises((RuntimeError, ImportError), match='vkjax_call'):
        hip.load_call_module()


def test_building_it_takes_pythons_headers(tmp_path, monkeypatch, capsys):
    monkeypatch.setattr(build, 'LIBDIR', str(tmp_path))
    monkeypatch.setattr(build.sysconfig, 'get_paths', lambda: {'include': str(tmp_path)})
    assert build.build_call() is None
    assert 'vkjax_call.so' in capsys.readouterr().out and not (tmp_path / 'vkjax_call.so').exists()
