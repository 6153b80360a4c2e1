'''How often planning looks at the launches of a program: a pass that has nothing to do there does not walk them. (CPU)'''
import numpy as np
import pytest

from vkjax_amd import fusion, minijax as mj, workloads as W
from vkjax_amd.jaxpr_interpreter import JaxprInterpreter


#looks at all launches together, as they were before passes for training steps and draws came in: no more than that
@pytest.mark.parametrize('name,most', [('affine', 18), ('conv_block', 58), ('mlp', 97)])
def test_looks_at_a_launch(name, most, monkeypatch):
    f, args = {'affine': (W.affine, W.affine_inputs()), 'conv_block': (W.conv_block, W.conv_block_inputs(batch=2, size=14, channels=16)),
               'mlp': (W.mlp, W.mlp_inputs())}[name]
    looks, reads = [0], fusion._reads
    def counted(op):
        looks[0] += 1
        return reads(op)
    monkeypatch.setattr(fusion, '_reads', counted)
    JaxprInterpreter(mj.make_jaxpr(f)(*args), plan_only=True)
    assert looks[0] <= most


def test_lists_that_a_pass_leaves_alone_stay_the_same_list():
    interp = JaxprInterpreter(mj.make_jaxpr(W.affine)(*W.affine_inputs()), plan_only=True)
    ops, pool = interp.all_ops, interp.bufferpool
    for name in ('fuse_softmax', 'fuse_row_programs', 'fuse_reduce_scales', 'fuse_reduce_updates', 'fuse_key_splits', 'fold_scalar_constants', 'remove_dead_ops'):
        assert getattr(fusion, name)(ops, pool, interp.jaxpr.jaxpr.outvars) is ops, name
    uses = fusion._use_counts(ops, pool, interp.jaxpr.jaxpr.outvars)
    assert fusion._use_counts(ops, pool, interp.jaxpr.jaxpr.outvars) is uses and fusion._use_counts(list(ops), pool, interp.jaxpr.jaxpr.outvars) == uses
