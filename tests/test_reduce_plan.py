'''Where a column sum of few rows is one launch and where two: both sides of every line. (CPU)'''
import pytest

from vkjax_amd import kernels as K


@pytest.mark.parametrize('rows,columns,one', [
    (1000, 10, True), (1536, 1000, True), (1537, 1000, False), (1536, 4096, True),
    #blocks that read 128 bytes of a row that begins anywhere in a line
    (1024, 5000, True), (1536, 4048, True), (1536, 4100, False), (1536, 5000, False), (1100, 7640, False), (1400, 5860, False), (1536, 4128, True),
    #large arrays in few blocks
    (900, 33216, False), (1536, 36864, False), (1536, 9408, True), (1536, 24576, True), (256, 65536, True),
    #read a word at a time
    (512, 4095, True), (1000, 4095, False)])
def test_lines(rows, columns, one):
    assert (K.plan_reduce_splits(1, rows, columns, 'reduce_sum') == 1) == one
