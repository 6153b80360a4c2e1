'''What a row program moves behind its launch still reads what it read where it stood. (CPU: the order of the launches)'''
import numpy as np
import pytest

from vkjax_amd import fusion, kernels as K, minijax as mj
from vkjax_amd.buffers import Buffer
from vkjax_amd.jaxpr_interpreter import JaxprInterpreter
from vkjax_amd.minijax import nn
from vkjax_amd.ops import Op


class Stop(Exception):
    pass


@pytest.mark.parametrize('written', ['read by the moved launch', 'something else'])
def test_a_later_write_follows_the_reader_that_moved(written, monkeypatch):
    '''reader = q + maxima of the first rows (moves: it reads a value of the program); writer changes q in place behind it.'''
    found = []
    def fuse(ops, bufferpool, outvars):
        at  = next(i for i, op in enumerate(ops) if fusion._is_row_reduction(op))
        top = ops[at].meta[1]
        q, other, out = (Buffer(None, np.float32, (4, 1)) for _ in range(3))
        whole  = lambda b: K.EwOperand(b, 0, (1, 1))
        reader = Op('reader', chain=K.EwChain(out, (4, 1), whole(q), [K.EwStep(K.EW['ADD_F'], whole(top))]))
        writer = Op('writer', launch=K.Launch('in_place', (1, 1, 1), (64, 1, 1), [(q if written.startswith('read') else other, 0)], b''))
        for op in (reader, writer):
            op.index = ops[at].index + 0.5
        result = original(ops[:at + 1] + [reader, writer] + ops[at + 1:], bufferpool, outvars)
        program = next(i for i, op in enumerate(result) if op.meta is not None and op.meta[0] == 'rows')
        found.extend([program, result.index(reader), result.index(writer)])
        indices = [op.index for op in result]
        assert indices == sorted(indices)
        raise Stop
    original = fusion.fuse_row_programs
    monkeypatch.setattr(fusion, 'fuse_row_programs', fuse)
    x = np.zeros((8, 10), np.float32)
    with pytest.raises(Stop):
        JaxprInterpreter(mj.make_jaxpr(lambda x: nn.log_softmax(x, axis=-1))(x), plan_only=True)
    program, reader, writer = found
    assert program < reader
    assert (reader < writer) if written.startswith('read') else (writer < program)
