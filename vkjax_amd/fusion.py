'''Peephole fusion over the op list of one program.

The reference issues one dispatch per jaxpr equation, plus one per implicit broadcast
(vkjax/kompute_jaxpr_interpreter.py:55-60, vkjax/ops.py:84-86), so a batch-norm + ReLU after a
convolution costs five full-size round trips through memory. Here two rewrites are applied
after the primitive dispatch and before storage is assigned:

  * chain + chain: an element-wise op whose input is the sole use of the previous element-wise
    op's full-size result continues that op's chain (one launch, intermediate never stored);
  * conv/dot + chain: add / sub / mul / div / max / min steps whose other operand is a scalar, a
    per-feature vector or a full-size tensor become the epilogue of the implicit-GEMM kernel and
    are applied to the accumulators before the only store.

Both keep the arithmetic and its order exactly as in the unfused program. A fused op sits at
the position of its last member, so the lifetimes of the earlier members' inputs are extended
to that position, and the skipped intermediates get no storage.
'''
import collections
import functools
import typing as tp

import numpy as np

from . import kernels as K
from .kernels import EW, EwChain, EwOperand, EwStep


class FusedEquation(tuple):
    '''Label of a fused op: the equations it covers, in order.'''
    def __repr__(self):
        return ' ; '.join(str(getattr(e, 'primitive', e)) for e in self)


_EPILOGUE_OPS = {EW[n] for n in ('ADD_F', 'SUB_F', 'MUL_F', 'DIV_F', 'MAX_F', 'MIN_F')}
_SELECTS      = {EW['SEL_P'], EW['SEL_T'], EW['SEL_F']}


def _reads(op) -> tp.List:
    '''Buffers an op reads (for plain launches: every buffer it touches).'''
    if op.chain is not None:
        return [o.buffer for o in op.chain.operands() if o is not None]
    if op.conv is not None:
        out, lhs, rhs, geom, epilogue = op.conv
        reads = [lhs, rhs] + [e.operand for e in epilogue if e.operand is not None and e.op not in (K.CONV_TAP, K.CONV_SOFTMAX)]
        for e in epilogue:
            reads += e.bounds
            if e.derived is not None:
                reads += [e.derived.first] + [st[1] for st in e.derived.steps if st[1] is not None]
        return reads
    if op.meta is not None:
        if op.meta[0] == 'iota':
            return []
        if op.meta[0] == 'concat_part':
            return [op.meta[2]]
        if op.meta[0] == 'threefry':
            return list(op.meta[2])
        if op.meta[0] == 'relu_backward':
            return [b for b, _ in op.launch.buffers[2:]]
        if op.meta[0] in ('random_stream', 'reduce', 'update', 'window_sum'):
            return [b for b, _ in op.launch.buffers[1:] if b is not None]
        if op.meta[0] == 'softmax':
            return [op.meta[2]]
        if op.meta[0] == 'rows':
            return list(op.meta[2])
        if op.meta[0] == 'conv_pack':
            return [op.meta[2].buffer]
    return [b for b, _ in op.launch.buffers if b is not None]


def _out(op):
    if op.chain is not None:
        return op.chain.out
    if op.conv is not None:
        return op.conv[0]
    return None


def _walks_densely(strides, shape) -> bool:
    '''The strides are the row-major ones of `shape`; the stride of a dimension of size 1 is never used and may be anything.'''
    return len(strides) == len(shape) and all(n == 1 or s == r for s, r, n in zip(strides, K.row_major_strides(shape), shape))


def _through_copy(operand: EwOperand, copy: EwChain, shape) -> tp.Optional[EwOperand]:
    '''`operand` (of a chain over `shape`) reads the result of `copy`, a chain without steps, i.e. result[c] =
    source[offset + c . strides] over copy.shape. When every dimension the operand walks is one dimension of the
    copy's result (a transposition, a slice, every n-th element, a broadcast of it, or the whole of it), the operand
    that reads the copy's source directly is returned: the two index maps composed. None otherwise.'''
    src, cshape = copy.first, tuple(copy.shape)
    if operand.buffer.size != np_prod(cshape) or len(operand.strides) != len(shape):
        return None
    dense = K.row_major_strides(cshape)
    rest, start = operand.offset, []
    for e in range(len(cshape)):
        start.append(rest // dense[e])
        rest -= start[-1] * dense[e]
    if rest:
        return None
    strides, taken = [], set()
    for n, s in zip(shape, operand.strides):
        if n == 1 or s == 0:
            strides.append(0)
            continue
        #the dimension with the largest pitch that divides the stride: the walk stays inside it or is none of one dimension
        dims = [e for e in range(len(cshape)) if cshape[e] > 1 and s > 0 and s % dense[e] == 0 and e not in taken]
        if not dims or start[dims[0]] + s // dense[dims[0]] * (n - 1) >= cshape[dims[0]]:
            return None
        taken.add(dims[0])
        strides.append(s // dense[dims[0]] * src.strides[dims[0]])
    return EwOperand(src.buffer, src.offset + sum(a * b for a, b in zip(start, src.strides)), tuple(strides))


def _is_full_contiguous(operand: EwOperand, shape) -> bool:
    return operand.offset == 0 and tuple(operand.buffer.shape) == tuple(shape) and _walks_densely(operand.strides, shape)


def _label(*ops):
    eqs = []
    for op in ops:
        eqs += list(op.equation) if isinstance(op.equation, FusedEquation) else [op.equation]
    return FusedEquation(eqs)


def _continuation_steps(chain: EwChain, producer_out) -> tp.Optional[tp.List[EwStep]]:
    '''The steps of `chain` re-expressed as a continuation of a chain that produced
    `producer_out`, or None if that value is not consumed as a plain full-size input exactly once.'''
    operands = chain.operands()
    hits = [k for k, o in enumerate(operands) if o is not None and o.buffer._placeholder is producer_out._placeholder]
    if len(hits) != 1:
        return None
    k = hits[0]
    if not _is_full_contiguous(operands[k], chain.shape):
        return None
    if k == 0:
        return list(chain.steps)
    if k == 1 and chain.steps[0].op not in _SELECTS and chain.steps[0].op != EW['NOP']:
        #acc = op(first, produced)  ->  acc = produced ; acc = op(first as operand on the other side, acc)
        s = chain.steps[0]
        return [EwStep(s.op, chain.first, not s.operand_left, s.imm)] + list(chain.steps[1:])
    return None


def _epilogue_steps(steps: tp.Sequence[EwStep], geom: K.ConvGeometry, out_shape) -> tp.Optional[tp.List[K.ConvEpilogueStep]]:
    result = []
    feature_dims = [d for d, s in enumerate(K.row_major_strides(out_shape)) if s == geom.os[3] and out_shape[d] == geom.N]
    for s in steps:
        if s.op not in _EPILOGUE_OPS or s.operand is None:
            return None
        o = s.operand
        if o.buffer.size == 1 and o.offset == 0:
            kind = 1
        elif _is_full_contiguous(o, out_shape):
            kind = 3
        elif (o.offset == 0 and o.buffer.size == geom.N and feature_dims
              and all((st == 1 if d == feature_dims[-1] else st == 0 or out_shape[d] == 1) for d, st in enumerate(o.strides))):
            kind = 2
        else:
            return None
        result.append(K.ConvEpilogueStep(s.op, kind, o.buffer, s.operand_left))
    return result


def _where(occurs):
    '''A pass that is entered only where an op it is about occurs, and hands the list it was given back where it changes
    nothing (what is known about a list of ops is kept with the list: _use_counts, remove_dead_ops).'''
    def only(fuse):
        @functools.wraps(fuse)
        def entered(ops, bufferpool, outvars):
            if not any(map(occurs, ops)):
                return ops
            result = fuse(ops, bufferpool, outvars)
            return ops if len(result) == len(ops) and all(a is b for a, b in zip(result, ops)) else result
        return entered
    return only


def _is(kind):
    return lambda op: op.meta is not None and op.meta[0] == kind


def fuse_ops(all_ops, bufferpool, outvars):
    from .ops import Op
    all_ops = fold_scalar_constants(all_ops, bufferpool, outvars)
    uses = collections.Counter()
    for op in all_ops:
        for b in _reads(op):
            uses[id(b._placeholder)] += 1
    for v in outvars:
        b = bufferpool.get_buffer(v)
        if b is not None:
            uses[id(b._placeholder)] += 2          #program outputs are never elided
            b.accesses.pop()                       #the lookup above is not a device access

    result: tp.List[tp.Optional[Op]] = []
    producer: tp.Dict[int, int] = {}               #placeholder id -> position in `result` of the op that wrote it
    last_reader: tp.Dict[int, int] = {}            #placeholder id -> position in `result` of the last op that read it

    def extend_lifetimes(op, index):
        for b in _reads(op):
            b.accesses.append(index)

    def fold_copies(op):
        '''An operand that is the full-size result of a pure copy (a broadcast, slice, transpose or reversal
        that was given a launch of its own) is read through that copy's strides instead; the copy goes away
        once nothing reads its result any more.'''
        chain, changed = op.chain, False
        first, steps = chain.first, list(chain.steps)
        for k, o in enumerate(chain.operands()):
            if o is None:
                continue
            pid = id(o.buffer._placeholder)
            pos = producer.get(pid)
            prod = result[pos] if pos is not None else None
            if prod is None or prod.chain is None or prod.chain.steps:
                continue
            source = _through_copy(o, prod.chain, chain.shape)
            if source is None:
                continue
            if k == 0:
                first = source
            else:
                steps[k - 1] = steps[k - 1]._replace(operand=source)
            changed = True
            uses[pid] -= 1
            uses[id(source.buffer._placeholder)] += 1
            source.buffer.accesses.append(op.index)
            if uses[pid] == 0:
                uses[id(source.buffer._placeholder)] -= 1
                _out(prod)._placeholder.elided = True
                result[pos] = None
                del producer[pid]
        if changed:
            new = Op(op.equation, chain=EwChain(chain.out, chain.shape, first, steps))
            new.index = op.index
            return new
        return op

    def conv_with_second_result(prod, op, pid):
        out, lhs, rhs, geom, epilogue = prod.conv
        #the merged launch stands where the chain stood: nothing in between may have read the convolution's result
        if last_reader.get(pid, -1) > producer[pid]:
            return None
        steps = _continuation_steps(op.chain, out)
        if steps is None or tuple(out.shape) != tuple(op.chain.shape) or op.chain.out.size != out.size:
            return None
        extra = _epilogue_steps(steps, geom, op.chain.shape)
        if extra is None or not K.conv_tap_supported(epilogue, extra) or K.conv_is_dense_rows(lhs, geom):
            return None
        tap = K.ConvEpilogueStep(K.CONV_TAP, 3, out)
        fused = Op(_label(prod, op), conv=(op.chain.out, lhs, rhs, geom, list(epilogue) + [tap] + extra))
        fused.index = op.index
        extend_lifetimes(prod, op.index)
        out.accesses.append(op.index)
        uses[pid] -= 1
        return fused

    def fold_pack_source(op):
        '''A kernel operand that is the result of a pure copy (the reversed kernel of an input gradient, a transposed
        weight matrix) is packed straight from that copy's source.'''
        _, packed, source, geom = op.meta
        pid = id(source.buffer._placeholder)
        prod = result[producer[pid]] if pid in producer else None
        if prod is None or prod.chain is None or prod.chain.steps:
            return op
        through = _through_copy(source, prod.chain, (geom.KH, geom.KW, geom.Cin, geom.N))
        if through is None:
            return op
        uses[pid] -= 1
        uses[id(through.buffer._placeholder)] += 1
        through.buffer.accesses.append(op.index)
        if uses[pid] == 0:
            uses[id(through.buffer._placeholder)] -= 1
            _out(prod)._placeholder.elided = True
            result[producer[pid]] = None
            del producer[pid]
        new = Op(op.equation, launch=K.conv_split_pack(packed, through, geom), meta=('conv_pack', packed, through, geom))
        new.index = op.index
        return new

    for op in all_ops:
        fused = None
        if op.meta is not None and op.meta[0] == 'conv_pack':
            op = fold_pack_source(op)
        if op.chain is not None:
            op = fold_copies(op)
            for cand in [o for o in op.chain.operands()[:2] if o is not None]:
                pid = id(cand.buffer._placeholder)
                pos = producer.get(pid)
                if pos is None or result[pos] is None:
                    continue
                prod = result[pos]
                if uses[pid] != 1:
                    #a convolution whose result something else reads as well can still take the chain over,
                    #by storing both: its result as it was, and the chain's
                    if prod.conv is not None and prod.conv[3].k_splits == 1 and _out(prod)._placeholder is cand.buffer._placeholder:
                        fused = conv_with_second_result(prod, op, pid)
                        if fused is not None:
                            result[pos] = None
                            break
                    continue
                steps = _continuation_steps(op.chain, _out(prod))
                if steps is None:
                    continue
                if prod.chain is not None:
                    if prod.chain.shape != op.chain.shape or 1 + len(prod.chain.steps) + len(steps) > K.EW_MAX_STEPS:
                        continue
                    chain = EwChain(op.chain.out, op.chain.shape, prod.chain.first, list(prod.chain.steps) + steps)
                    fused = Op(_label(prod, op), chain=chain)
                else:
                    out, lhs, rhs, geom, epilogue = prod.conv
                    if geom.k_splits > 1 or tuple(out.shape) != tuple(op.chain.shape) or len(epilogue) + len(steps) > K.CONV_MAX_EPI:
                        continue
                    extra = _epilogue_steps(steps, geom, op.chain.shape)
                    if extra is None:
                        continue
                    if geom.shares is not None and not K.conv_straight_epilogue(list(epilogue) + extra):
                        continue                                  #(the kernels whose blocks share tiles have no other)
                    if not K.conv_epilogue_is_worth_leaving_four_waves(lhs, rhs, geom, list(epilogue) + extra):
                        continue
                    if K.conv_is_dense_rows(lhs, geom) and not K.dense_rows_epilogue_supported(list(epilogue) + extra):
                        continue                                  #the chain stays a launch of its own
                    tap_at = [k for k, e in enumerate(epilogue) if e.op == K.CONV_TAP]
                    if tap_at and not K.conv_tap_supported(epilogue[:tap_at[0]], list(epilogue[tap_at[0] + 1:]) + extra):
                        continue
                    fused = Op(_label(prod, op), conv=(op.chain.out, lhs, rhs, geom, list(epilogue) + extra))
                fused.index = op.index
                extend_lifetimes(prod, op.index)
                _out(prod)._placeholder.elided = True
                result[pos] = None
                del producer[pid]
                break
        new = fused if fused is not None else op
        result.append(new)
        for b in _reads(new):
            last_reader[id(b._placeholder)] = len(result) - 1
        out = _out(new)
        if out is not None:
            producer[id(out._placeholder)] = len(result) - 1
        else:
            #a launch that is neither a chain nor a convolution may change its result buffer in place (scatter-add
            #accumulates into a copy of its operand): whoever produced that buffer before no longer describes what
            #it holds, so nothing behind this launch may be joined to that producer or read through it
            for b in _writes(new):
                producer.pop(id(b._placeholder), None)
    ops = fuse_random_streams([op for op in result if op is not None], bufferpool, outvars)
    ops = fuse_key_splits(remove_dead_ops(fuse_stream_chains(ops, bufferpool, outvars), bufferpool, outvars), bufferpool, outvars)
    ops = fuse_softmax(ops, bufferpool, outvars)
    ops = fuse_row_programs(remove_dead_ops(ops, bufferpool, outvars), bufferpool, outvars)
    ops = fuse_scale_relu_backward(ops, bufferpool, outvars)
    ops = fuse_reduce_prologues(ops, bufferpool, outvars)
    ops = fuse_reduce_scales(ops, bufferpool, outvars)
    ops = fuse_reduce_updates(ops, bufferpool, outvars)
    ops = fuse_derived_epilogue_operands(ops, bufferpool, outvars)
    ops = fuse_relu_backward_epilogues(ops, bufferpool, outvars)
    ops = fuse_window_sums(ops, bufferpool, outvars)
    ops = fuse_relu_backward_sums(ops, bufferpool, outvars)
    ops = fuse_index_wrap(ops, bufferpool, outvars)
    ops = fold_index_wrap(ops, bufferpool, outvars)
    ops = fuse_dense_softmax(ops, bufferpool, outvars)
    ops = remove_dead_ops(ops, bufferpool, outvars)
    bufferpool.use_counts, bufferpool.without_dead = (None, None), None
    return batch_small_chains(batch_packs(ops))


@_where(_is('reduce'))
def fuse_softmax(ops, bufferpool, outvars):
    '''softmax over the last dimension as jax.nn.softmax spells it,

        m = reduce_max(x) ; e = exp(x - m) ; s = reduce_sum(e) ; y = e / s

    becomes one launch when m, e and s are used by nothing else. Same values, bit for bit: the fused kernel
    adds in the order of the row reduction it replaces.'''
    from .ops import Op
    uses = _use_counts(ops, bufferpool, outvars)
    pid  = lambda b: id(b._placeholder)
    removed, replacement = set(), {}

    def per_row(operand, shape):
        return (operand is not None and operand.offset == 0 and len(shape) >= 1
                and tuple(operand.strides) == K.row_major_strides(shape[:-1] + (1,))[:-1] + (0,))

    for i, R1 in enumerate(ops):
        if R1.meta is None or R1.meta[0] != 'reduce' or i + 3 >= len(ops):
            continue
        _, m, x, outer, rows, inner, name, _, nsplit = R1.meta
        C1, R2, C2 = ops[i + 1], ops[i + 2], ops[i + 3]
        if (name != 'reduce_max' or inner != 1 or nsplit != 1 or x.dtype != 'float32' or not 0 < rows < K.SOFTMAX_MAX_ROW
                or C1.chain is None or C2.chain is None or R2.meta is None or R2.meta[0] != 'reduce'):
            continue
        c1, c2 = C1.chain, C2.chain
        _, s, e, outer2, rows2, inner2, name2, _, nsplit2 = R2.meta
        flat = lambda shape: (int(np_prod(shape[:-1])), shape[-1]) if len(shape) else (1, 1)
        if (name2 != 'reduce_sum' or (outer2, rows2, inner2, nsplit2) != (outer, rows, 1, 1)
                or flat(c1.shape) != (outer, rows) or flat(c2.shape) != (outer, rows)
                or c1.first.buffer._placeholder is not x._placeholder or not _is_full_contiguous_any_shape(c1.first, c1.shape)
                or [st.op for st in c1.steps] != [EW['SUB_F'], EW['EXP_F']] or c1.steps[0].operand_left
                or c1.steps[0].operand.buffer._placeholder is not m._placeholder or not per_row(c1.steps[0].operand, c1.shape)
                or e._placeholder is not c1.out._placeholder
                or c2.first.buffer._placeholder is not c1.out._placeholder or not _is_full_contiguous_any_shape(c2.first, c2.shape)
                or [st.op for st in c2.steps] != [EW['DIV_F']] or c2.steps[0].operand_left
                or c2.steps[0].operand.buffer._placeholder is not s._placeholder or not per_row(c2.steps[0].operand, c2.shape)
                or uses[pid(m)] != 1 or uses[pid(c1.out)] != 2 or uses[pid(s)] != 1):
            continue
        members, last, arg_out = (R1, C1, R2, C2), C2, None
        #the arg-max over the same rows of the probabilities, right behind them: one more result of the same launch
        A = ops[i + 4] if i + 4 < len(ops) else None
        if (A is not None and A.meta is not None and A.meta[0] == 'reduce' and A.meta[6] == 'argmax' and A.meta[8] == 1
                and A.meta[2]._placeholder is c2.out._placeholder and tuple(A.meta[3:6]) == (outer, rows, 1) and A.meta[1].dtype == 'int32'):
            members, last, arg_out = (R1, C1, R2, C2, A), A, A.meta[1]
            removed.add(i + 3)
        fused = Op(_label(*members), launch=K.softmax_rows(c2.out, x, outer, rows, arg_out),
                   meta=('softmax', [c2.out] + ([arg_out] if arg_out is not None else []), x, outer, rows))
        fused.index = last.index
        x.accesses.append(last.index)
        if arg_out is not None:
            c2.out.accesses.append(last.index)
        for b in (m, c1.out, s):
            b._placeholder.elided = True
        removed |= {i, i + 1, i + 2}
        replacement[i + 3 + (arg_out is not None)] = fused
    return [replacement.get(i, op) for i, op in enumerate(ops) if i not in removed]


#From three ops on a launch is saved whatever else the step needs. There is no upper line to the array's size: a loss and its
#gradient on rows of 10, 64, 100, 256, 1000 and 1001 were faster in one launch on 50 to 262144 rows, where they take 36 to 838 us
#through the separate launches (1000 x 10: 39 -> 16 us, 65536 x 64: 120 -> 56, 65536 x 1000: 838 -> 462).
ROW_PROGRAM_MIN_OPS = 3


def _row_walk(operand: EwOperand, shape, outer: int, R: int):
    '''(element of row 0, row stride, column stride, one value per row) of an operand of a chain over `shape`, an array of
    [outer, R] or of `outer` values, or None where its rows do not lie at one stride.'''
    full = len(shape) > 0 and shape[-1] == R and np_prod(shape) == outer * R
    if not full and np_prod(shape) != outer:
        return None
    walk  = list(zip(shape, operand.strides))
    outer_dims = [(n, s) for n, s in (walk[:-1] if full else walk) if n != 1]
    for (_, s), (m, t) in zip(outer_dims, outer_dims[1:]):
        if s != t * m:
            return None
    return operand.offset, outer_dims[-1][1] if outer_dims else 0, walk[-1][1] if full else 0, not full


class _RowProgram:
    '''The instructions of a run of row-wise ops (`members`, in order), or no `launch` where they do not fit the kernel.'''

    def __init__(self, members, outer: int, R: int, needed_outside):
        pid = lambda b: id(b._placeholder)
        self.inputs, self.outs, self.steps, self.inside, self.launch = [], [], [], {}, None
        result_of = lambda op: op.meta[1] if op.chain is None else op.chain.out
        made      = {pid(result_of(op)): n for n, op in enumerate(members)}
        self.inside = {pid(result_of(op)): result_of(op) for op in members}
        singles, number, in_acc, in_slots = {}, {}, None, set()

        def operand(o: EwOperand, shape):
            '''(slot, one value per row) an operand is read from; None: it is not read as the kernel reads.'''
            walk = _row_walk(o, shape, outer, R)
            if walk is None:
                return None
            base, row, column, whole_row = walk
            if pid(o.buffer) in made:
                single = singles.get(pid(o.buffer))
                if single is None or (base, row, column) != (0, 1 if single else R, 0 if single or whole_row else 1) or (whole_row and not single):
                    return None
                return ('value', pid(o.buffer)), single
            i = K.RowsInput(o.buffer, base, row, column, column == 0)
            if i not in self.inputs:
                self.inputs.append(i)
            return ('in', self.inputs.index(i)), i.single

        #values that a later member reads otherwise than from the accumulator the moment they are made
        reads = []
        for op in members:
            o = [EwOperand(op.meta[2], 0, (R, 1))] if op.chain is None else op.chain.operands()
            reads.append([None if x is None else pid(x.buffer) for x in o])
        keep = set()
        for n, r in enumerate(reads):
            for k, b in enumerate(r):
                if b in made and not (k == 0 and made[b] == n - 1):
                    keep.add(b)

        def load(o, shape):
            nonlocal in_acc
            where = operand(o, shape)
            if where is None:
                return False
            if where[0] != ('value', in_acc):
                self.steps.append(K.RowsStep('load', slot=where[0], single=where[1]))
            return True

        for op in members:
            if op.chain is None:
                _, out, source, _, _, _, name, _, _ = op.meta
                if not load(EwOperand(source, 0, (R, 1)), (outer, R)):
                    return
                self.steps.append(K.RowsStep(name))
                single = True
            else:
                chain = op.chain
                out   = chain.out
                if any(s.op in _SELECTS for s in chain.steps) or not load(chain.first, chain.shape):
                    return
                for s in chain.steps:
                    where = (None, False)
                    if s.operand is not None:
                        where = operand(s.operand, chain.shape)
                        if where is None:
                            return
                    self.steps.append(K.RowsStep('apply', s.op, s.operand_left, where[0], where[1], s.imm))
                single = np_prod(chain.shape) != outer * R
            singles[pid(out)] = single
            in_acc = pid(out)
            if pid(out) in keep:
                self.steps.append(K.RowsStep('put', slot=('value', pid(out)), single=single))
            if pid(out) in needed_outside:
                self.steps.append(K.RowsStep('out', slot=('out', len(self.outs)), single=single))
                self.outs.append(out)
        self.launch = K.row_program(self.outs, self.inputs, self.steps, outer, R)


@_where(lambda op: _is_row_reduction(op))
def fuse_row_programs(ops, bufferpool, outvars):
    '''Element-wise chains and row reductions over the rows of one [outer, R] array that feed each other - a classifier's
    loss and its gradient - become one launch (rows.hip), values bit for bit. What stands between them and reads
    their results moves behind it.'''
    from .ops import Op
    pid  = lambda b: id(b._placeholder)
    done = set()
    while True:
        seed = next((i for i, op in enumerate(ops) if id(op) not in done and _is_row_reduction(op)), None)
        if seed is None:
            return ops
        done.add(id(ops[seed]))
        _, _, _, outer, R, _, _, _, _ = ops[seed].meta
        program, members, behind = _row_program_around(ops, seed, outer, R, bufferpool, outvars)
        if program is None:
            continue
        last  = members[-1]
        fused = Op(_label(*[ops[i] for i in members]), launch=program.launch, meta=('rows', program.outs, [i.buffer for i in program.inputs]))
        fused.index = ops[last].index
        for b in [i.buffer for i in program.inputs] + program.outs:
            b.accesses.append(fused.index)
        for key, b in program.inside.items():
            if not any(pid(o) == key for o in program.outs):
                b._placeholder.elided = True
        #what moves gets a place of its own between the launch and whatever followed it
        for n, i in enumerate(behind):
            ops[i].index = fused.index + (n + 1) / (len(behind) + 1)
            for b in _touched(ops[i]) + [b for b, _ in ops[i].launch.buffers if b is not None]:
                b.accesses.append(ops[i].index)
        taken = set(members) | set(behind)
        ops = ([op for i, op in enumerate(ops[:last]) if i not in taken] + [fused] + [ops[i] for i in behind] + list(ops[last + 1:]))


def _is_row_reduction(op) -> bool:
    if op.meta is None or op.meta[0] != 'reduce' or op.chain is not None or op.conv is not None:
        return False
    _, _, source, outer, R, inner, name, _, nsplit = op.meta
    return (inner == 1 and nsplit == 1 and name in ('reduce_sum', 'reduce_max') and source.dtype == np.float32
            and 2 <= R <= K.ROWS_MAX_ROW and outer >= 2 and outer * R < 2**30)


def _row_program_around(ops, seed: int, outer: int, R: int, bufferpool, outvars):
    '''(program, positions of its members, positions of the ops among them that move behind it) for the largest run of ops
    connected to the reduction at `seed`, or (None, ...).'''
    pid = lambda b: id(b._placeholder)

    def candidate(op) -> bool:
        if _is_row_reduction(op):
            return op.meta[3:5] == (outer, R)
        if op.chain is None or op.meta is not None or np_prod(op.chain.shape) not in (outer, outer * R):
            return False
        return all(o is None or (o.buffer.size < 2**30 and _row_walk(o, op.chain.shape, outer, R) is not None) for o in op.chain.operands())

    result_of  = lambda op: op.meta[1] if op.chain is None else op.chain.out
    candidates = [i for i, op in enumerate(ops) if candidate(op)]
    #connected through the values they make
    maker, group = {pid(result_of(ops[i])): i for i in candidates}, {seed}
    while True:
        more = {i for i in candidates if i not in group
                and (any(maker.get(pid(b)) in group for b in _reads(ops[i])) or any(maker.get(pid(b)) == i for g in group for b in _reads(ops[g])))}
        if not more:
            break
        group |= more
    members = sorted(group)
    counts  = collections.Counter(pid(b) for op in ops for b in _writes(op))
    while len(members) >= ROW_PROGRAM_MIN_OPS:
        inside, tainted, wanted, taken, behind = set(), set(), set(), [], []
        for i in range(members[0], members[-1] + 1):
            op = ops[i]
            if i in members and not any(pid(b) in tainted for b in _reads(op)) and counts[pid(result_of(op))] == 1:
                taken.append(i)
                inside.add(pid(result_of(op)))
            elif any(pid(b) in tainted or pid(b) in inside for b in _touched(op)) or any(pid(b) in wanted for b in _written(op)):
                #(what it reads may not be written in front of it either)
                behind.append(i)
                tainted |= {pid(b) for b in _may_write(op)}
                wanted  |= {pid(b) for b in _reads(op)}
        if len(taken) < ROW_PROGRAM_MIN_OPS or seed not in taken:
            return None, [], []
        if taken != members:
            members = taken
            continue
        #nothing that stands behind a member and in front of the launch may change what the member reads
        read = set()
        for i in range(members[0], members[-1] + 1):
            if i in members:
                read |= {pid(b) for b in _reads(ops[i])}
            elif any(pid(b) in read or pid(b) in inside for b in _may_write(ops[i])):
                return None, [], []
        uses = _use_counts(ops, bufferpool, outvars)
        own  = collections.Counter(pid(b) for i in members for b in _reads(ops[i]))
        program = _RowProgram([ops[i] for i in members], outer, R, {k for k in inside if uses[k] > own[k]})
        if program.launch is not None:
            return program, members, [i for i in behind if i < members[-1]]
        members = members[:-1] if members[-1] != seed else members[1:]
    return None, [], []


@_where(lambda op: op.chain is not None and len(op.chain.steps) == 3 and op.chain.steps[0].op == EW['LT_I'])
def fuse_index_wrap(ops, bufferpool, outvars):
    '''`select(x < 0, x + n, x)` on int32, the way tracing normalises an index that may count from the end, is two
    launches after chain fusion (x + n, and the comparison with the select, which needs x + n as a second full-size
    value). One opcode does it in one pass over x.'''
    from .ops import Op
    uses = _use_counts(ops, bufferpool, outvars)
    pid  = lambda b: id(b._placeholder)
    writer = {pid(op.chain.out): i for i, op in enumerate(ops) if op.chain is not None}
    same   = lambda a, b: a.buffer._placeholder is b.buffer._placeholder and a.offset == b.offset and tuple(a.strides) == tuple(b.strides)
    single = lambda o: o is not None and all(s == 0 for s in o.strides)
    removed, replacement = set(), {}
    for i, B in enumerate(ops):
        ch = B.chain
        if ch is None or [st.op for st in ch.steps] != [EW['LT_I'], EW['SEL_P'], EW['NOP']]:
            continue
        less, pick, carrier = ch.steps
        zero = getattr(less.operand.buffer, 'constant_value', None) if single(less.operand) else None
        if (less.operand_left or zero is None or np_prod(zero.shape) != 1 or int(zero.reshape(-1)[0]) != 0
                or not same(carrier.operand, ch.first) or not _is_full_contiguous_any_shape(pick.operand, ch.shape)):
            continue
        a = writer.get(pid(pick.operand.buffer))
        if a is None or a >= i or a in removed or uses[pid(pick.operand.buffer)] != 1:
            continue
        A = ops[a].chain
        if (tuple(A.shape) != tuple(ch.shape) or len(A.steps) != 1 or A.steps[0].op != EW['ADD_I'] or not single(A.steps[0].operand)
                or not same(A.first, ch.first) or A.out.dtype != ch.first.buffer.dtype):
            continue
        fused = Op(_label(ops[a], B), chain=EwChain(ch.out, ch.shape, ch.first, [EwStep(EW['WRAP_I'], A.steps[0].operand)]))
        fused.index = B.index
        A.steps[0].operand.buffer.accesses.append(B.index)
        pick.operand.buffer._placeholder.elided = True
        removed.add(a)
        replacement[i] = fused
    return [replacement.get(i, op) for i, op in enumerate(ops) if i not in removed]


@_where(lambda op: op.chain is not None and len(op.chain.steps) == 1 and op.chain.steps[0].op == EW['WRAP_I'])
def fold_index_wrap(ops, bufferpool, outvars):
    '''The normalised copy of an index array, `select(i < 0, i + n, i)` (one launch after fuse_index_wrap), is not made
    when everything that reads it is a row gather or a sorted row scatter-add: those kernels read the indices as they
    are and add n to the negative ones themselves.'''
    from .ops import Op
    uses = _use_counts(ops, bufferpool, outvars)
    pid  = lambda b: id(b._placeholder)
    removed, replacement = set(), {}
    for i, op in enumerate(ops):
        ch = op.chain
        if ch is None or len(ch.steps) != 1 or ch.steps[0].op != EW['WRAP_I'] or ch.steps[0].operand_left:
            continue
        o = ch.steps[0].operand
        amount = getattr(o.buffer, 'constant_value', None) if o is not None and all(st == 0 for st in o.strides) else None
        if (amount is None or np_prod(amount.shape) != 1 or not _is_full_contiguous_any_shape(ch.first, ch.shape)
                or str(ch.first.buffer.dtype) != 'int32' or str(ch.out.dtype) != 'int32'):
            continue
        readers = [j for j in range(len(ops)) if j != i and any(b._placeholder is ch.out._placeholder for b in _reads(ops[j]))]
        if not readers or len(readers) != uses[pid(ch.out)] or min(readers) < i:
            continue                                           #(also a result of the program: its uses count two more)
        ok = True
        for j in readers:
            r = replacement.get(j, ops[j])
            where = K.INDEX_WRAP_KERNELS.get(r.launch.kernel) if r.chain is None and r.conv is None else None
            places = [k for k, (b, _) in enumerate(r.launch.buffers) if b is not None and b._placeholder is ch.out._placeholder] if where else []
            ok = ok and where is not None and places == [where[0]]
        #the raw indices must still be what they were where the readers run
        last = max(readers)
        if not ok or any(w._placeholder is ch.first.buffer._placeholder for j in range(i + 1, last + 1) for w in _may_write(ops[j])):
            continue
        for j in readers:
            r = replacement.get(j, ops[j])
            launch = K.with_wrapped_index(r.launch, ch.first.buffer, ch.first.offset * 4, int(amount.reshape(-1)[0]))
            new = Op(_label(op, r), launch=launch, meta=r.meta)
            new.index = r.index
            ch.first.buffer.accesses.append(r.index)
            replacement[j] = new
        ch.out._placeholder.elided = True
        removed.add(i)
    return [replacement.get(i, op) for i, op in enumerate(ops) if i not in removed]


@_where(_is('softmax'))
def fuse_dense_softmax(ops, bufferpool, outvars):
    '''A classifier's last layer: a product with at most 16 output features, read by nothing but the softmax launch
    right behind it, computes the softmax (and the arg-max that launch carries) on the row before it is stored
    (dense_rows_n16). The exponentials are added in the order of the separate launch: same values, bit for bit.'''
    from .ops import Op
    uses = _use_counts(ops, bufferpool, outvars)
    removed, replacement = set(), {}
    for i, (D, S) in enumerate(zip(ops, ops[1:])):
        if D.conv is None or S.meta is None or S.meta[0] != 'softmax':
            continue
        out, lhs, rhs, geom, epilogue = D.conv
        _, results, x, outer, rows = S.meta
        if (x._placeholder is not out._placeholder or uses[id(out._placeholder)] != 1 or (geom.M, geom.N) != (outer, rows)
                or any(e.op in (K.CONV_TAP, K.CONV_SOFTMAX) for e in epilogue)):
            continue
        steps = list(epilogue) + [K.ConvEpilogueStep(K.CONV_SOFTMAX, 0, results[1] if len(results) > 1 else None)]
        try:
            K.conv_gemm(results[0], lhs, rhs, geom, steps)
        except ValueError:
            continue                                   #another kernel serves this product
        fused = Op(_label(D, S), conv=(results[0], lhs, rhs, geom, steps))
        fused.index = S.index
        for b in _reads(D):
            b.accesses.append(S.index)
        out._placeholder.elided = True
        removed.add(i)
        replacement[i + 1] = fused
    return [replacement.get(i, op) for i, op in enumerate(ops) if i not in removed]


def np_prod(values) -> int:
    out = 1
    for v in values:
        out *= int(v)
    return out


@_where(_is('reduce'))
def fuse_reduce_prologues(ops, bufferpool, outvars):
    '''A float column sum whose operand is, and is only, the result of `a * b` (b of the same shape or a
    vector over the columns) or of `-a` reads a (and b) itself and applies the step while loading: the
    pairs `multiply -> reduce_sum` and `negate -> reduce_sum` of a batch-norm backward pass lose a full-size
    array each. Values are unchanged (same products, same order of additions).'''
    from .ops import Op
    uses = _use_counts(ops, bufferpool, outvars)
    pid  = lambda b: id(b._placeholder)
    chain_writer = {pid(op.chain.out): i for i, op in enumerate(ops) if op.chain is not None}
    removed, replacement = set(), {}
    for i, R in enumerate(ops):
        if R.meta is None or R.meta[0] != 'reduce':
            continue
        _, out, inp, outer, rows, inner, name, partial, nsplit = R.meta
        w = chain_writer.get(pid(inp))
        if name != 'reduce_sum' or inner <= 1 or inp.dtype != 'float32' or w is None or w > i or w in removed or uses[pid(inp)] != 1:
            continue
        ch = ops[w].chain
        size = 1
        for d in ch.shape:
            size *= d
        if size != outer * rows * inner or len(ch.steps) != 1 or not _is_full_contiguous_any_shape(ch.first, ch.shape):
            continue
        step, prologue = ch.steps[0], None
        if step.op == EW['NEG_F'] and step.operand is None:
            prologue = ('neg', None)
        elif step.op == EW['MUL_F'] and step.operand is not None:
            o = step.operand
            if _is_full_contiguous_any_shape(o, ch.shape):
                prologue = ('mul', o.buffer)
            elif (o.offset == 0 and o.buffer.size == inner and ch.shape[-1] == inner
                  and tuple(o.strides) == (0,) * (len(ch.shape) - 1) + (1,)):
                prologue = ('mulv', o.buffer)
        if prologue is None:
            continue
        source = ch.first.buffer
        launch = K.reduce(out, source, outer, rows, inner, name, partial, nsplit, prologue=prologue)[0]
        fused  = Op(_label(ops[w], R), launch=launch, meta=None)
        fused.index = R.index
        for b in (source, prologue[1]):
            if b is not None:
                b.accesses.append(R.index)
        ch.out._placeholder.elided = True
        removed.add(w)
        replacement[i] = fused
    return [replacement.get(i, op) for i, op in enumerate(ops) if i not in removed]


def _is_float_sum(op) -> bool:
    '''A launch that writes finished float sums: an unsplit reduction, or the second launch of one that is split (of the
    slices of a kernel gradient too).'''
    return (op.chain is None and op.conv is None and (op.meta is None or op.meta[0] == 'reduce')
            and op.launch.kernel.startswith(('reduce_rows_fsum_v', 'reduce_cols_fsum_v')))


def _sole_reader_takes(ops, i, C, uses) -> bool:
    '''The sum ops[i], which ops[C] reads, is read by nothing else and could be taken where ops[C] stands: its operand still
    holds the same values there.'''
    out, source = ops[i].launch.buffers[0][0], ops[i].launch.buffers[1][0]
    #(a launch without a record of its structure counts among the readers of its own result)
    own = sum(b._placeholder is out._placeholder for b in _reads(ops[i]))
    return (i < C and uses[id(out._placeholder)] - own == 1
            and not any(w._placeholder is source._placeholder for j in range(i + 1, C) for w in _written(ops[j])))


@_where(_is('reduce'))
def fuse_reduce_scales(ops, bufferpool, outvars):
    '''A float sum (one launch: not split into ranges) whose result is read once, by `sum / c`, `sum * c` or `-(sum / c)` with a single value c - a mean, a mean
    negative log-likelihood - stores that itself: the element-wise launch behind it goes away. The division is the one
    the element-wise kernel would have made (same operands, same rounding).'''
    from .ops import Op
    uses = _use_counts(ops, bufferpool, outvars)
    pid  = lambda b: id(b._placeholder)
    sums = {pid(op.launch.buffers[0][0]): i for i, op in enumerate(ops) if _is_float_sum(op) and op.meta is not None and op.meta[8] == 1}
    removed, replacement = set(), {}
    for C, op in enumerate(ops):
        ch = op.chain
        if ch is None or not ch.steps or ch.steps[0].operand is None:
            continue
        kind = {(EW['DIV_F'],): 'div', (EW['MUL_F'],): 'times', (EW['DIV_F'], EW['NEG_F']): 'negdiv'}.get(tuple(st.op for st in ch.steps))
        total, o = ch.first, ch.steps[0].operand
        if kind == 'times' and pid(total.buffer) not in sums:
            total, o = o, ch.first                              #c * sum: the product is the same number
        i = sums.get(pid(total.buffer))
        if (kind is None or (kind != 'times' and ch.steps[0].operand_left) or i is None or not _sole_reader_takes(ops, i, C, uses)
                or not _is_full_contiguous_any_shape(total, ch.shape) or o.buffer.size != 1 or o.offset != 0
                or o.buffer.dtype != 'float32' or ch.out.dtype != 'float32' or ch.out.size != total.buffer.size):
            continue
        launch = K.sum_with_post(ops[i].launch, ch.out, kind, o.buffer)
        if launch is None:
            continue
        fused = Op(_label(ops[i], op), launch=launch, meta=None)
        fused.index = op.index
        for b in (ops[i].launch.buffers[1][0], o.buffer):
            b.accesses.append(op.index)
        total.buffer._placeholder.elided = True
        removed.add(i)
        replacement[C] = fused
    return [replacement.get(i, op) for i, op in enumerate(ops) if i not in removed]


@_where(lambda op: _is_float_sum(op))
def fuse_reduce_updates(ops, bufferpool, outvars):
    '''A float column sum (of the slices of a kernel gradient, of the rows of a bias gradient) whose result is read once, by
    `p - rate * sum` with a single value `rate` - a step of gradient descent - stores that difference itself. Same
    operands and roundings as the element-wise launch behind it, which goes away. There is no lower or upper line: it is one
    launch, one write and one read of the gradient less at every size (a training step of a 784-300-100-10 network over 1000
    rows 145 -> 128 us together with its weight gradients in the layout of the weights, ResNet-50's 12.82 -> 12.74 ms).'''
    from .ops import Op
    uses = _use_counts(ops, bufferpool, outvars)
    pid  = lambda b: id(b._placeholder)
    sums = {pid(op.launch.buffers[0][0]): i for i, op in enumerate(ops) if _is_float_sum(op)}
    removed, replacement = set(), {}
    for C, op in enumerate(ops):
        ch = op.chain
        if ch is None or [st.op for st in ch.steps] != [EW['MUL_F'], EW['SUB_F']] or not ch.steps[1].operand_left:
            continue
        total, rate, before = ch.first, ch.steps[0].operand, ch.steps[1].operand
        if pid(total.buffer) not in sums:
            total, rate = rate, total                           #rate * sum: the product is the same number
        i = sums.get(pid(total.buffer))
        if i is None or not _sole_reader_takes(ops, i, C, uses):
            continue
        n = total.buffer.size
        if (rate.buffer.size != 1 or rate.offset != 0 or ch.out.size != n or before.buffer.size != n or before.buffer.dtype != 'float32'
                or ch.out.dtype != 'float32' or not all(_is_full_contiguous_any_shape(o, ch.shape) for o in (total, before))):
            continue
        launch = K.column_sum_update(ops[i].launch, ch.out, before.buffer, rate.buffer)
        if launch is None:
            continue
        fused = Op(_label(ops[i], op), launch=launch, meta=('update',))
        fused.index = op.index
        ops[i].launch.buffers[1][0].accesses.append(op.index)
        total.buffer._placeholder.elided = True
        removed.add(i)
        replacement[C] = fused
    return [replacement.get(i, op) for i, op in enumerate(ops) if i not in removed]


@_where(_is('reduce'))
def fuse_scale_relu_backward(ops, bufferpool, outvars):
    '''The backward pass of a per-channel scale and shift followed by ReLU (a batch norm with fixed statistics
    and its activation), as reverse-mode differentiation emits it:

        m = select(ans > t, g, z) ; db = sum_rows(m) ; dx = m * k ; p = m * x ; dk = sum_rows(p)

    with m read by nothing else and p only by its sum, becomes ONE launch that reads ans, g and x once and
    writes dx and both column sums (their first stage, when the sums are split over row ranges). The sums are
    taken in the order of the reduce_cols launches they replace, so every value keeps its bits.'''
    from .ops import Op
    uses = _use_counts(ops, bufferpool, outvars)
    pid  = lambda b: id(b._placeholder)
    last_writer: tp.Dict[int, int] = {}
    for i, op in enumerate(ops):
        for b in _may_write(op):
            last_writer[pid(b)] = i
    readers: tp.Dict[int, tp.List[int]] = {}
    for i, op in enumerate(ops):
        for b in _reads(op):
            readers.setdefault(pid(b), []).append(i)
    single = lambda o: o is not None and o.offset == 0 and all(st == 0 for st in o.strides)
    removed, replacement = set(), {}

    def column_sum_of(i, buffer):
        '''(rows, inner, nsplit) when ops[i] is the float sum over the rows of `buffer` seen as [rows, inner].'''
        R = ops[i]
        if R.meta is None or R.meta[0] != 'reduce':
            return None
        _, out, inp, outer, rows, inner, name, partial, nsplit = R.meta
        if (name != 'reduce_sum' or outer != 1 or inner <= 1 or inp.dtype != 'float32' or inp._placeholder is not buffer._placeholder
                or rows * inner != buffer.size or not R.launch.kernel.startswith('reduce_cols_fsum_v')):
            return None
        return rows, inner, nsplit

    def select_chain(op):
        ch = op.chain
        return (ch is not None and [st.op for st in ch.steps] == [EW['GT_F'], EW['SEL_P'], EW['NOP']] and not ch.steps[0].operand_left
                and single(ch.steps[0].operand) and single(ch.steps[2].operand)
                and _is_full_contiguous_any_shape(ch.first, ch.shape) and _is_full_contiguous_any_shape(ch.steps[1].operand, ch.shape)
                and ch.out.dtype == 'float32' and ch.first.buffer.dtype == 'float32')

    chain_writer = {pid(op.chain.out): i for i, op in enumerate(ops) if op.chain is not None}
    for R1, first_sum in enumerate(ops):
        if first_sum.meta is None or first_sum.meta[0] != 'reduce':
            continue
        m = first_sum.meta[2]
        geometry = column_sum_of(R1, m)
        if geometry is None:
            continue
        rows, inner, nsplit = geometry
        C, P = None, None
        #several such backward passes can share one m (two branches of a residual block): each sum
        #goes with the first scaling and the first product that follow it
        for r in sorted(readers.get(pid(m), [])):
            other = ops[r].chain
            if r < R1 or other is None or [st.op for st in other.steps] != [EW['MUL_F']] or other.shape[-1] != inner or other.out.size != m.size:
                continue
            a, b = other.first, other.steps[0].operand
            if b is not None and a.buffer._placeholder is not m._placeholder:
                a, b = b, a
            if b is None or a.buffer._placeholder is not m._placeholder or not _is_full_contiguous_any_shape(a, other.shape):
                continue
            if _is_full_contiguous_any_shape(b, other.shape) and b.buffer.dtype == 'float32':
                P = P or (r, b.buffer)
            elif (b.offset == 0 and b.buffer.size == inner and b.buffer.dtype == 'float32'
                  and tuple(b.strides) == (0,) * (len(other.shape) - 1) + (1,)):
                C = C or (r, b.buffer)
        if C is None or P is None or C[0] == P[0]:
            continue
        p_out = ops[P[0]].chain.out
        R2 = [r for r in readers.get(pid(p_out), []) if column_sum_of(r, p_out) is not None]
        if uses[pid(p_out)] != 1 or len(R2) != 1 or column_sum_of(R2[0], p_out) != geometry:
            continue
        R2 = R2[0]
        if ops[R1].launch.kernel != ops[R2].launch.kernel or ops[R1].launch.params != ops[R2].launch.params:
            continue
        x, k = P[1], C[1]
        # with the select: where the select stood, if the three launches above are all that read its result
        M = chain_writer.get(pid(m))
        with_select = M is not None and M < min(R1, C[0], P[0]) and select_chain(ops[M]) and uses[pid(m)] == 3
        position = M if with_select else min(R1, C[0], P[0])
        involved = [R1, C[0], P[0], R2] + ([M] if with_select else [])
        if any(j in removed or j in replacement for j in involved):
            continue
        #everything the merged launch reads has to exist where the first of the launches it replaces stood
        sources = [x, k] + ([o.buffer for o in ops[M].chain.operands()] if with_select else [m])
        if any(last_writer.get(pid(b), -1) >= position for b in sources):
            continue
        dx, sum_m, sum_mx = ops[C[0]].chain.out, ops[R1].launch.buffers[0][0], ops[R2].launch.buffers[0][0]
        if with_select:
            ch = ops[M].chain
            launch = K.scale_relu_backward(ops[R1].launch, dx, sum_m, sum_mx, x, k, ch.steps[1].operand.buffer,
                                           select=(ch.first.buffer, ch.steps[0].operand.buffer, ch.steps[2].operand.buffer))
            m._placeholder.elided = True
        else:
            launch = K.scale_relu_backward(ops[R1].launch, dx, sum_m, sum_mx, x, k, m)
        fused = Op(_label(*[ops[j] for j in sorted(involved)]), launch=launch)
        fused.index = ops[position].index
        for b, _ in launch.buffers:
            if b is not None:
                b.accesses.append(fused.index)
        p_out._placeholder.elided = True
        removed |= set(involved) - {position}
        replacement[position] = fused
    return [replacement.get(i, op) for i, op in enumerate(ops) if i not in removed]


def fuse_relu_backward_epilogues(ops, bufferpool, outvars):
    '''The backward pass of a ReLU behind a product on the bf16 matrix cores (the gradient of a layer's input, to which another
    branch's may have been added) and the scaling in front of that ReLU,

        d = product (+ r) ; m = select(ans > t, d, z) ; dx = m * k

    with d read by nothing else, become the product's epilogue. Where m is read elsewhere too it is the launch's second result.
    The arithmetic and its order are unchanged. The merged launch stands where the select stood.'''
    from .ops import Op
    if not any(op.conv is not None and op.conv[3].split is not None for op in ops):
        return ops
    uses   = _use_counts(ops, bufferpool, outvars)
    pid    = lambda b: id(b._placeholder)
    single = lambda o: o is not None and o.buffer.size == 1 and o.offset == 0 and o.buffer.dtype == 'float32'
    ops    = list(ops)
    maker  = {pid(op.conv[0]): i for i, op in enumerate(ops) if op.conv is not None and op.conv[3].split is not None}
    last_writer: tp.Dict[int, int] = {}
    readers: tp.Dict[int, tp.List[int]] = {}
    for i, op in enumerate(ops):
        for b in _written(op):
            last_writer[pid(b)] = i
        for b in _reads(op):
            readers.setdefault(pid(b), []).append(i)

    def scaling(chain, shape, geom):
        '''(scaled buffer, epilogue step) of a chain that only multiplies by a value per feature.'''
        if chain is None or [st.op for st in chain.steps] != [EW['MUL_F']] or tuple(chain.shape) != tuple(shape) or chain.steps[0].operand is None:
            return None
        for a, b in ((chain.first, chain.steps[0].operand), (chain.steps[0].operand, chain.first)):
            step = _epilogue_steps([EwStep(EW['MUL_F'], b)], geom, shape)
            if _is_full_contiguous(a, shape) and step is not None and step[0].kind == 2:
                return a.buffer, step[0]
        return None

    for i, op in enumerate(ops):
        ch = op.chain if op is not None else None
        if (ch is None or [st.op for st in ch.steps[:3]] != [EW['GT_F'], EW['SEL_P'], EW['NOP']] or ch.steps[0].operand_left or len(ch.steps) > 4
                or not single(ch.steps[0].operand) or not single(ch.steps[2].operand) or ch.out.dtype != 'float32' or ch.first.buffer.dtype != 'float32'
                or not _is_full_contiguous(ch.first, ch.shape) or not _is_full_contiguous(ch.steps[1].operand, ch.shape)):
            continue
        d, activation = ch.steps[1].operand.buffer, ch.first.buffer
        at = maker.get(pid(d))
        if at is None or at >= i or uses[pid(d)] != 1 or ops[at] is None or pid(activation) == pid(d):
            continue
        out, lhs, rhs, geom, epilogue = ops[at].conv
        if tuple(out.shape) != tuple(ch.shape) or ch.out.size != out.size or activation.size != out.size:
            continue
        #what the product reads still has to be there where the select stood
        if any(last_writer.get(pid(b), -1) > at and pid(b) != pid(d) for b in _reads(ops[at])):
            continue
        steps = list(epilogue) + [K.ConvEpilogueStep(K.CONV_MASK, 3, activation, bounds=(ch.steps[0].operand.buffer, ch.steps[2].operand.buffer))]
        result, involved = ch.out, [at, i]
        if len(ch.steps) == 4:
            vector = _epilogue_steps(ch.steps[3:], geom, ch.shape)
            if vector is None:
                continue
            steps += vector
        else:
            for r in sorted(readers.get(pid(ch.out), [])):
                scaled = scaling(ops[r].chain, ch.shape, geom) if r > i and ops[r] is not None else None
                if scaled is not None and pid(scaled[0]) == pid(ch.out) and last_writer.get(pid(scaled[1].operand), -1) < i:
                    steps += [K.ConvEpilogueStep(K.CONV_TAP, 3, ch.out), scaled[1]]
                    result, involved = ops[r].chain.out, [at, i, r]
                    break
        if K.conv_masked_epilogue(steps) is None:
            continue
        fused = Op(_label(*[ops[j] for j in involved]), conv=(result, lhs, rhs, geom, steps))
        fused.index = op.index
        for b in _reads(fused) + _writes(fused):
            b.accesses.append(fused.index)
        d._placeholder.elided = True
        for j in involved:
            ops[j] = None
        ops[i] = fused
    return [op for op in ops if op is not None]


def _select_by_threshold(chain) -> bool:
    '''`chain` is select(ans > t, g, z) of two whole float arrays and two single values.'''
    single = lambda o: o is not None and o.offset == 0 and o.buffer.size == 1 and o.buffer.dtype == 'float32'
    return (chain is not None and [st.op for st in chain.steps] == [EW['GT_F'], EW['SEL_P'], EW['NOP']] and not chain.steps[0].operand_left
            and single(chain.steps[0].operand) and single(chain.steps[2].operand)
            and all(_is_full_contiguous_any_shape(o, chain.shape) and o.buffer.dtype == 'float32' for o in (chain.first, chain.steps[1].operand))
            and chain.out.dtype == 'float32' and chain.out.size == np_prod(chain.shape))


@_where(_is('reduce'))
def fuse_relu_backward_sums(ops, bufferpool, outvars):
    '''The backward pass of a dense layer's ReLU and the gradient of the bias in front of it,

        m = select(ans > t, g, z) ; db = sum_rows(m)

    become ONE launch that writes m and the column sums (their first stage, when they are split over row ranges), in the order
    of the launch it replaces. It runs behind the passes that take the select into a product's epilogue and those that let an
    unsplit sum store an updated parameter: what is left are gradients that are results of the program and, in a training step, sums of
    more rows than one launch takes. No line by size: the launch has the grid of the sum, and replays of the pair alone took as long or
    longer at every size that was timed (127 x 256 14.6 -> 5.4 us, 1000 x 300 18.4 -> 15.3, 1000 x 7 15.2 -> 15.4, 65536 x 256 52.4 ->
    42.9, 100000 x 33 30.4 -> 29.4).'''
    from .ops import Op
    pid = lambda b: id(b._placeholder)
    selects = {pid(op.chain.out): i for i, op in enumerate(ops) if _select_by_threshold(op.chain)}
    removed, replacement = set(), {}
    for i, R in enumerate(ops):
        if R.meta is None or R.meta[0] != 'reduce' or R.launch.kernel not in K.REDUCE_BATCH_KERNELS:
            continue
        _, _, m, outer, rows, inner, _, _, _ = R.meta
        M = selects.get(pid(m))
        if M is None or M > i or M in replacement or outer != 1 or rows * inner != m.size:
            continue
        ch, sums = ops[M].chain, R.launch.buffers[0][0]
        #the sums are written where the select stood, and m must not change between there and the launch that summed it
        if any(pid(b) in (pid(m), pid(sums)) for op in ops[M + 1:i] for b in _may_write(op)):
            continue
        launch = K.relu_backward(R.launch, ch.out, sums, ch.steps[1].operand.buffer, (ch.first.buffer, ch.steps[0].operand.buffer, ch.steps[2].operand.buffer))
        fused  = Op(_label(ops[M], R), launch=launch, meta=('relu_backward', [ch.out, sums]))
        fused.index = ops[M].index
        for b, _ in launch.buffers:
            b.accesses.append(fused.index)
        removed.add(i)
        replacement[M] = fused
    return [replacement.get(i, op) for i, op in enumerate(ops) if i not in removed]


def fuse_window_sums(ops, bufferpool, outvars):
    '''Average pooling and its gradient: float sums under windows over [batch, y, x, channels] take over, where nothing else reads
    the arrays in between,

        the pad with zeros that spreads their operand (the gradient under strided windows), and in front of it or of the sum
        a division or multiplication by one value, of a whole array or of one value per image and channel;
        behind the sum, a division or multiplication by one value or the selection select(ans > t, sum, z)

    Same values added in the same order, and the same roundings. The merged launch stands where the last of those stood. No line by
    size: a pooling with one scaling takes one launch for two, 2.7 us instead of 5.4 on 2 x 8 x 8 x 16 and 38 instead of 61 to 105 on 64 x 56
    x 56 x 256.'''
    from .ops import Op
    uses = _use_counts(ops, bufferpool, outvars)
    pid  = lambda b: id(b._placeholder)
    name = lambda op: getattr(getattr(op.equation, 'primitive', None), 'name', '') if op.chain is None and op.conv is None and op.meta is None else ''
    if not any(name(op) == 'reduce_window_sum' for op in ops):
        return ops
    single = lambda o: o is not None and o.offset == 0 and o.buffer.size == 1 and o.buffer.dtype == 'float32'
    ops    = list(ops)
    #(a plain launch counts among the readers of its own result)
    read_once = lambda i, b: uses[pid(b)] - sum(r._placeholder is b._placeholder for r in _reads(ops[i])) == 1
    maker = {}
    for i, op in enumerate(ops):
        out = _out(op) if op.chain is not None else op.launch.buffers[0][0] if name(op) == 'pad' else None
        if out is not None:
            maker[pid(out)] = i

    def scaling(chain, of=None):
        '''(the scaled operand, ('div' | 'times', value)) of a chain of that one step (of the buffer `of`), or (None, None).'''
        if len(chain.steps) == 1 and chain.steps[0].operand is not None and chain.out.dtype == 'float32':
            step = chain.steps[0]
            for scaled, value in ((chain.first, step.operand), (step.operand, chain.first)):
                if not single(value) or scaled.buffer.dtype != 'float32' or (of is not None and scaled.buffer._placeholder is not of._placeholder):
                    continue
                if step.op == EW['MUL_F']:                       #value * x: the product is the same number
                    return scaled, ('times', value.buffer)
                if step.op == EW['DIV_F'] and step.operand_left == (scaled is step.operand):
                    return scaled, ('div', value.buffer)
        return None, None

    for w, W in enumerate(ops):
        if W is None or name(W) != 'reduce_window_sum' or not W.launch.kernel.startswith('pool2d_') or W.launch.buffers[1][0].dtype != 'float32':
            continue
        out, source = W.launch.buffers[0][0], W.launch.buffers[1][0]
        params = W.equation.params
        if len(source.shape) != 4 or tuple(out.shape) != tuple(W.equation.outvars[0].aval.shape):
            continue
        at       = lambda seq: tuple(int(v) for v in seq[1:3])
        low      = at([p[0] for p in params['padding']])
        members, before, after, spread = [w], None, None, (1, 1)
        #the pad with zeros
        i = maker.get(pid(source))
        if i is not None and i < w and ops[i] is not None and name(ops[i]) == 'pad' and read_once(i, source):
            P     = ops[i]
            value = P.launch.buffers[2][0].constant_value
            config = [tuple(int(v) for v in c) for c in P.equation.params['padding_config']]
            if (value is not None and np.asarray(value).size == 1 and np.asarray(value, np.float32).tobytes() == bytes(4) and len(config) == 4
                    and config[0] == config[3] == (0, 0, 0) and all(v >= 0 for c in config[1:3] for v in c)):
                members.append(i)
                low    = tuple(l + c[0] for l, c in zip(low, config[1:3]))
                spread = tuple(c[2] + 1 for c in config[1:3])
                source = P.launch.buffers[1][0]
        extent  = tuple(source.shape[1:3])
        operand = EwOperand(source, 0, K.row_major_strides(source.shape))
        #a scaling in front
        i = maker.get(pid(source))
        if i is not None and i < w and ops[i] is not None and ops[i].chain is not None and read_once(i, source):
            ch = ops[i].chain
            scaled, before = scaling(ch)
            #(a division is repeated for every window an element lies in: left alone where that may be nine times)
            taps = K._cdiv(int(params['window_dimensions'][1]), spread[0]) * K._cdiv(int(params['window_dimensions'][2]), spread[1])
            if before is not None and tuple(ch.shape) == tuple(source.shape) and (taps <= 4 or before[0] == 'times'):
                members.append(i)
                operand = scaled
            else:
                before = None
        #what follows
        position = w
        reader = [j for j in range(w + 1, len(ops)) if ops[j] is not None and any(b._placeholder is out._placeholder for b in _reads(ops[j]))]
        if len(reader) == 1 and ops[reader[0]].chain is not None and read_once(w, out):
            ch = ops[reader[0]].chain
            if _select_by_threshold(ch) and ch.steps[1].operand.buffer._placeholder is out._placeholder and ch.first.buffer._placeholder is not out._placeholder:
                after = ('select', ch.steps[0].operand.buffer, ch.steps[2].operand.buffer, ch.first.buffer)
            else:
                scaled, after = scaling(ch, of=out)
                if after is not None and not _is_full_contiguous_any_shape(scaled, ch.shape):
                    after = None
            if after is not None:
                position = reader[0]
                members.append(position)
        if len(members) == 1:
            continue
        result = ops[position].chain.out if after is not None else out
        if result.size != out.size:
            continue
        #(the result may carry another shape: the launch is laid out by the windows')
        shaped = result if tuple(result.shape) == tuple(out.shape) else result.view(result.dtype, out.shape)
        launch = K.pool_sum(shaped, operand, extent, low, spread, at(params['window_dimensions']), at(params['window_strides']),
                            at(params.get('window_dilation') or (1,) * 4), before, after)
        if launch is None:
            continue
        reads = [b for b, _ in launch.buffers[1:] if b is not None and b.constant_value is None]
        if any(w_._placeholder is b._placeholder for j in range(min(members) + 1, position) if j not in members and ops[j] is not None
               for w_ in _may_write(ops[j]) for b in reads):
            continue
        fused = Op(_label(*[ops[j] for j in sorted(members)]), launch=launch, meta=('window_sum',))
        fused.index = ops[position].index
        for b, _ in launch.buffers:
            if b is not None:
                b.accesses.append(fused.index)
        for j in members:
            if j != position:
                (_out(ops[j]) if ops[j].chain is not None else ops[j].launch.buffers[0][0])._placeholder.elided = True
                ops[j] = None
        ops[position] = fused
    return [op for op in ops if op is not None]


@_where(lambda op: op.chain is not None and op.chain.out.size == 1 and op.chain.out.tensor is None)
def fold_scalar_constants(ops, bufferpool, outvars):
    '''Arithmetic on single floats that are known when the program is built (-1 / 1000, the factor of a mean's gradient) is done
    then, with the device's rounding, and its result is a constant like the ones it came from: one launch less per value
    (4 us in a chain of small launches). Results that are no normal number or zero are left to the device.'''
    from .buffers import to_device_words
    operations = {EW['NEG_F']: lambda a, b: -a, EW['ADD_F']: lambda a, b: a + b, EW['SUB_F']: lambda a, b: a - b,
                  EW['MUL_F']: lambda a, b: a * b, EW['DIV_F']: lambda a, b: a / b}
    returned = set()
    for v in outvars:
        b = bufferpool.get_buffer(v)
        if b is not None:
            returned.add(id(b._placeholder))
            b.accesses.pop()                       #the lookup above is not a device access
    normal   = lambda v: v == 0 or (np.isfinite(v) and abs(v) >= np.finfo(np.float32).tiny)

    def known(operand):
        b = operand.buffer
        if b.size != 1 or b.dtype != 'float32' or operand.offset != 0 or b.constant_value is None:
            return None
        value = np.asarray(b.constant_value)
        return np.float32(value.reshape(())) if value.size == 1 and value.dtype in (np.float32, np.float64) else None

    kept = []
    for op in ops:
        ch = op.chain
        if (ch is None or ch.out.size != 1 or ch.out.dtype != 'float32' or not ch.steps or ch.out.tensor is not None
                or id(ch.out._placeholder) in returned or any(st.op not in operations for st in ch.steps)):
            kept.append(op)
            continue
        value = known(ch.first)
        for st in ch.steps:
            other = known(st.operand) if st.operand is not None else np.float32(0)
            if value is None or other is None:
                value = None
                break
            with np.errstate(all='ignore'):
                value = operations[st.op](*((other, value) if st.operand_left else (value, other)))
            value = value if normal(value) else None
        if value is None:
            kept.append(op)
            continue
        ch.out.tensor         = bufferpool.device.tensor(to_device_words(value.reshape(1)))
        ch.out.constant_value = value
        ch.out.accesses      += [0, np.inf]
    return kept


def _is_full_contiguous_any_shape(operand: EwOperand, shape) -> bool:
    '''The operand covers `shape` densely in row-major order (its buffer may carry another shape of the same size).'''
    size = 1
    for d in shape:
        size *= d
    return operand.offset == 0 and operand.buffer.size == size and _walks_densely(operand.strides, shape)


@_where(_is('random_stream'))
def fuse_stream_chains(ops, bufferpool, outvars):
    '''A launch that generates random words (random_bits lowered directly) followed by an
    element-wise chain over exactly those words whose operands are single values: the chain is
    applied by the generating kernel before its only store.'''
    from .ops import Op
    uses = _use_counts(ops, bufferpool, outvars)
    pid  = lambda b: id(b._placeholder)
    removed, replacement = set(), {}
    for si, S in enumerate(ops):
        if S.meta is None or S.meta[0] != 'random_stream':
            continue
        _, out, layout, key0, key1, h, c0, c1, n, steps = S.meta[:10]
        if layout == 'pairs' or uses[pid(out)] != 1 or steps:
            continue
        for i in range(si + 1, len(ops)):
            op = ops[i]
            if not any(b._placeholder is out._placeholder for b in _reads(op)):
                continue
            ch = op.chain
            size = 1
            for d in (ch.shape if ch is not None else ()):
                size *= d
            if (ch is not None and ch.first.buffer._placeholder is out._placeholder and ch.first.offset == 0 and size == out.size
                    and tuple(ch.first.strides) == K.row_major_strides(ch.shape) and len(ch.steps) <= K.TF_MAX_STEPS
                    and all(st.op not in _SELECTS and st.op != EW['NOP'] and
                            (st.operand is None or (st.operand.buffer.size == 1 and st.operand.offset == 0)) for st in ch.steps)):
                fused = Op(_label(S, op), launch=K.threefry_stream(ch.out, key0, key1, h, c0, c1, list(ch.steps), layout=layout, n=n),
                           meta=('random_stream', ch.out, layout, key0, key1, h, c0, c1, n, list(ch.steps)))
                fused.index = op.index
                for b in [key0[0], key1[0]] + [st.operand.buffer for st in ch.steps if st.operand is not None]:
                    b.accesses.append(fused.index)
                out._placeholder.elided = True
                removed.add(si)
                replacement[i] = fused
            break
    return [replacement.get(i, op) for i, op in enumerate(ops) if i not in removed]


@_where(_is('random_stream'))
def fuse_key_splits(ops, bufferpool, outvars):
    '''A key split (a launch of random words without steps) whose words nothing but the keys of other draws read: those draws
    compute their two words of it themselves. Same bits; the split's launch goes.'''
    from .ops import Op
    uses = _use_counts(ops, bufferpool, outvars)
    pid  = lambda b: id(b._placeholder)
    writers = collections.defaultdict(list)
    for i, op in enumerate(ops):
        for b in _may_write(op):
            writers[pid(b)].append(i)
    result, gone = list(ops), set()
    #(from the end: a split that a draw has taken over may itself read the words of another)
    for si in reversed(range(len(ops))):
        S = result[si]
        if S.meta is None or S.meta[0] != 'random_stream' or si in gone:
            continue
        if len(S.meta) > 10:
            continue
        _, out, layout, key0, key1, h, c0, c1, n, steps = S.meta
        if steps or layout == 'xor':
            continue
        reading = lambda b: [i for i in range(len(ops)) if i != si and i not in gone and any(r._placeholder is b._placeholder for r in _reads(result[i]))]
        #where the words are read: from the split's result itself, or from a copy of one key of it
        places, copies = [(out, 0, 1)], []
        for i in reading(out):
            ch = result[i].chain
            if ch is not None and not ch.steps and ch.out.size == 2 and max(ch.shape) == 2 and len(writers[pid(ch.out)]) == 1:
                places.append((ch.out, ch.first.offset, ch.first.strides[list(ch.shape).index(2)]))
                copies.append(i)
        takes = lambda op, b: (op.meta is not None and op.meta[0] == 'random_stream' and len(op.meta) == 10
                               and all(k[0]._placeholder is b._placeholder for k in op.meta[3:5])
                               and sum(r._placeholder is b._placeholder for r in _reads(op)) == 2)
        draws = [(i, first, step) for b, first, step in places for i in reading(b) if i not in copies]
        if (not draws or min(i for i, _, _ in draws) < si or len(writers[pid(out)]) != 1
                or not all(takes(result[i], b) for b, _, _ in places for i in reading(b) if i not in copies)
                or any(uses[pid(b)] != 2 * len([i for i in reading(b) if i not in copies]) + (len(copies) if b is out else 0) for b, _, _ in places)
                or any(writers[pid(k[0])] and max(writers[pid(k[0])]) > si for k in (key0, key1))):
            continue
        for i, first, step in draws:
            op = result[i]
            _, out2, layout2, (_, w0), (_, w1), h2, d0, d1, n2, steps2 = op.meta
            split = K.KeySplit(layout, h, c0, c1, 2 * h if layout == 'pairs' else n, (first + w0 * step, first + w1 * step))
            fused = Op(_label(S, op), launch=K.threefry_stream(out2, key0, key1, h2, d0, d1, steps2, layout=layout2, n=n2, key_split=split),
                       meta=('random_stream', out2, layout2, key0, key1, h2, d0, d1, n2, steps2, split))
            fused.index = op.index
            for b in (key0[0], key1[0]):
                b.accesses.append(fused.index)
            result[i] = fused
        for i in copies:
            result[i].chain.out._placeholder.elided = True
            gone.add(i)
        out._placeholder.elided = True
        gone.add(si)
    return [op for i, op in enumerate(result) if i not in gone]


@_where(lambda op: op.conv is not None and any(e.kind == 2 and e.derived is None for e in op.conv[4]))
def fuse_derived_epilogue_operands(ops, bufferpool, outvars):
    '''A per-feature operand of a convolution epilogue that is itself the result of a short chain over
    per-feature vectors and single values (the batch-norm scale gamma * rsqrt(var + eps)) is computed
    by the convolution kernel while it stages its epilogue operands; the chain's own launch and its
    result array go away. One such operand per convolution; the arithmetic is unchanged.'''
    from .ops import Op
    uses = _use_counts(ops, bufferpool, outvars)
    pid  = lambda b: id(b._placeholder)
    producer = {pid(op.chain.out): i for i, op in enumerate(ops) if op.chain is not None}
    allowed  = {EW[name] for name in K.CONV_DERIVED_OPS}
    unary    = {EW['NEG_F'], EW['RSQRT_F'], EW['SQRT_F']}
    removed  = set()
    result   = list(ops)
    for ci, op in enumerate(ops):
        if op.conv is None:
            continue
        out, lhs, rhs, geom, epilogue = op.conv
        N = geom.N
        if K.conv_is_dense_rows(lhs, geom):
            continue                                              #that kernel reads its epilogue operands as they are
        for ei, e in enumerate(epilogue):
            if e.kind != 2 or e.derived is not None or e.operand is None:
                continue
            pi = producer.get(pid(e.operand))
            if pi is None or pi >= ci or pi in removed or uses[pid(e.operand)] != 1:
                continue
            chain = ops[pi].chain
            n = 1
            for d in chain.shape:
                n *= d
            if n != N or not (1 <= len(chain.steps) <= K.CONV_MAX_DERIVED):
                continue

            def per_feature(o):
                '''(buffer) if the operand is one value or walks N contiguous values, else None'''
                if o.offset != 0:
                    return None
                if o.buffer.size == 1:
                    return o.buffer
                if o.buffer.size == N and tuple(o.strides) == K.row_major_strides(chain.shape):
                    return o.buffer
                return None
            first = per_feature(chain.first)
            steps = []
            for st in chain.steps:
                if st.op not in allowed or st.imm:
                    steps = None
                    break
                if st.op in unary:
                    if st.operand is not None:
                        steps = None
                        break
                    steps.append((st.op, None, False))
                else:
                    b = per_feature(st.operand) if st.operand is not None else None
                    if b is None:
                        steps = None
                        break
                    steps.append((st.op, b, bool(st.operand_left)))
            if first is None or steps is None:
                continue
            derived  = K.ConvDerivedOperand(first, tuple(steps))
            new_epi  = list(epilogue)
            new_epi[ei] = e._replace(operand=None, derived=derived)
            fused = Op(_label(ops[pi], op), conv=(out, lhs, rhs, geom, new_epi))
            fused.index = op.index
            for b in [first] + [st[1] for st in steps if st[1] is not None]:
                b.accesses.append(fused.index)
            e.operand._placeholder.elided = True
            removed.add(pi)
            result[ci] = fused
            break
    return [op for i, op in enumerate(result) if i not in removed]


def _writes(op) -> tp.List:
    if op.conv is not None:
        return [_out(op)] + [e.operand for e in op.conv[4] if e.op in (K.CONV_TAP, K.CONV_SOFTMAX) and e.operand is not None]
    if op.chain is not None:
        return [_out(op)]
    if op.meta is not None and op.meta[0] in ('iota', 'concat_part'):
        return [op.meta[1]]
    if op.meta is not None and op.meta[0] in ('threefry', 'softmax', 'rows', 'relu_backward'):
        return list(op.meta[1])
    return [b for b, _ in op.launch.buffers[:1] if b is not None]      #kernels write their first argument


def remove_dead_ops(ops, bufferpool, outvars):
    '''Drops launches none of whose results is read by a later launch or returned (the unused half
    of a PRNG key split, for instance). The reference runs every equation; the values returned
    are the same.'''
    while bufferpool.without_dead is not ops:
        uses = _use_counts(ops, bufferpool, outvars)
        #an accumulating kernel (scatter-add) also reads what it writes: such a use does not keep it alive
        dead = {i for i, op in enumerate(ops)
                if _writes(op) and all(uses[id(b._placeholder)] - sum(1 for r in _reads(op) if r._placeholder is b._placeholder) == 0
                                       for b in _writes(op))
                and not any(sum(1 for o in ops if any(w._placeholder is b._placeholder for w in _writes(o))) > 1 for b in _writes(op))}
        if not dead:
            bufferpool.without_dead = ops
            break
        for i in dead:
            for b in _writes(ops[i]):
                b._placeholder.elided = True
        ops = [op for i, op in enumerate(ops) if i not in dead]
    return ops


def _use_counts(ops, bufferpool, outvars):
    '''How often every array is read by the ops of this list, two more for results of the program; not to be changed. Kept
    until another list is asked about: the passes do not change the lists they are given.'''
    counted, uses = bufferpool.use_counts
    if counted is ops:
        return uses
    uses = collections.Counter()
    for op in ops:
        for b in _reads(op):
            uses[id(b._placeholder)] += 1
    for v in outvars:
        b = bufferpool.get_buffer(v)
        if b is not None:
            uses[id(b._placeholder)] += 2
            b.accesses.pop()
    bufferpool.use_counts = (ops, uses)
    return uses


@_where(_is('threefry'))
def fuse_random_streams(ops, bufferpool, outvars):
    '''Collapses the random-bits pipeline into one launch:

        c = iota(2h); a, b = threefry2x32(key, c[:h], c[h:]); bits = concatenate(a, b); out = chain(bits)

    where `chain` is an element-wise chain whose operands are single values (jax.random.uniform's
    shift / or / bitcast / sub / mul / add / max). The fused kernel generates the counters in
    registers and applies the chain before its only store, so of the iota, the two slices, the
    block function, the two concatenate copies and the chain only one write of the result remains.
    The arithmetic per element is unchanged. A draw of an odd number of words n = 2h - 1 has c = concatenate(iota(n), 0) and drops
    the last of the bits, which the kernel does itself.'''
    from .ops import Op
    uses = collections.Counter(_use_counts(ops, bufferpool, outvars))      #(counted down below)
    pid  = lambda b: id(b._placeholder)
    writers = collections.defaultdict(list)          #placeholder id -> positions of the ops that write it
    for i, op in enumerate(ops):
        if op.chain is not None or op.conv is not None:
            writers[pid(_out(op))].append(i)
        elif op.meta is not None and op.meta[0] == 'iota':
            writers[pid(op.meta[1])].append(i)
        elif op.meta is not None and op.meta[0] == 'concat_part':
            writers[pid(op.meta[1])].append(i)
        elif op.meta is not None and op.meta[0] == 'threefry':
            for b in op.meta[1]:
                writers[pid(b)].append(i)
        else:
            for b, _ in op.launch.buffers[:1]:       #kernels write their first argument
                if b is not None:
                    writers[pid(b)].append(i)
    def padded(ws, counters) -> bool:
        '''Whether the two launches at `ws` write an iota of 2h - 1 words and a zero behind it.'''
        if len(ws) != 2 or len(counters.shape) != 1 or counters.dtype != 'uint32' or any(ops[i].meta is None or ops[i].meta[0] != 'concat_part' for i in ws):
            return False
        (_, _, words, d0, at0, *_), (_, _, pad, d1, at1, *_) = sorted((ops[i].meta for i in ws), key=lambda m: m[4])
        source = writers.get(pid(words), [])
        return ((d0, at0, d1, at1) == (0, 0, 0, words.size) and pad.size == 1 and counters.size == words.size + 1 and words.size > 1 and words.dtype == 'uint32'
                and pad.dtype == 'uint32' and pad.constant_value is not None and int(np.asarray(pad.constant_value).reshape(())) == 0 and not writers.get(pid(pad))
                and len(source) == 1 and ops[source[0]].meta is not None and ops[source[0]].meta[0] == 'iota' and len(words.shape) == 1)

    removed = set()
    replacement = {}
    for ti, T in enumerate(ops):
        if T.meta is None or T.meta[0] != 'threefry' or not T.meta[3]:
            continue
        (aa, ab), (key0, key1, x0, x1), _ = T.meta[1:]
        h = x0.size
        if aa.size != h or len(aa.shape) != 1:
            continue
        #counters: contiguous slices of one-dimensional uint32 iotas
        sources = []
        for xb in (x0, x1):
            w = writers.get(pid(xb), [])
            if len(w) != 1 or uses[pid(xb)] != 1:
                break
            C = ops[w[0]]
            if C.chain is None or C.chain.steps or len(C.chain.shape) != 1 or tuple(C.chain.first.strides) != (1,):
                break
            S  = C.chain.first.buffer
            ws = writers.get(pid(S), [])
            if padded(ws, S):
                sources.append((w[0], C.chain.first.offset, ws, S))
                continue
            if len(ws) != 1 or ops[ws[0]].meta is None or ops[ws[0]].meta[0] != 'iota' or len(S.shape) != 1 or S.dtype != 'uint32':
                break
            sources.append((w[0], C.chain.first.offset, ws[0], S))
        if len(sources) != 2:
            continue
        odd = [isinstance(ws, list) for _, _, ws, _ in sources]
        if any(odd) and not (all(odd) and sources[0][3]._placeholder is sources[1][3]._placeholder and uses[pid(sources[0][3])] == 2
                             and sources[0][3].size == 2 * h and (sources[0][1], sources[1][1]) == (0, h)):
            continue
        count = 2 * h - 1 if any(odd) else 2 * h
        #results: concatenated in order into one array
        if uses[pid(aa)] != 1 or uses[pid(ab)] != 1:
            continue
        cats = [i for i, op in enumerate(ops) if op.meta is not None and op.meta[0] == 'concat_part'
                and op.meta[2]._placeholder in (aa._placeholder, ab._placeholder)]
        if len(cats) != 2:
            continue
        m0, m1 = ops[cats[0]].meta, ops[cats[1]].meta
        if m0[2]._placeholder is not aa._placeholder:
            m0, m1 = m1, m0
        AC = m0[1]
        if (m0[2]._placeholder is not aa._placeholder or m1[2]._placeholder is not ab._placeholder or m1[1]._placeholder is not AC._placeholder
                or len(AC.shape) != 1 or AC.size != 2 * h or (m0[3], m0[4], m1[3], m1[4]) != (0, 0, 0, h)
                or sorted(writers[pid(AC)]) != sorted(cats)):
            continue
        #an element-wise chain on the bits whose operands are single values
        chain_pos = None
        if uses[pid(AC)] == 1:
            for i in range(max(cats) + 1, len(ops)):
                op = ops[i]
                if any(b._placeholder is AC._placeholder for b in _reads(op)):
                    ch = op.chain
                    n  = 1
                    for d in (ch.shape if ch is not None else ()):
                        n *= d
                    if (ch is not None and ch.first.buffer._placeholder is AC._placeholder and ch.first.offset == 0 and n == count
                            and tuple(ch.first.strides) == K.row_major_strides(ch.shape) and len(ch.steps) <= K.TF_MAX_STEPS
                            and all(st.op not in _SELECTS and st.op != EW['NOP'] and
                                    (st.operand is None or (st.operand.buffer.size == 1 and st.operand.offset == 0)) for st in ch.steps)):
                        chain_pos = i
                    break
        if any(odd) and chain_pos is None:
            continue
        members = [sources[0][0], sources[1][0], ti] + cats + ([chain_pos] if chain_pos is not None else []) + (sources[0][2] if any(odd) else [])
        if removed & set(members):
            continue
        last  = max(members)
        out   = ops[chain_pos].chain.out if chain_pos is not None else AC
        steps = list(ops[chain_pos].chain.steps) if chain_pos is not None else []
        #a key word that is a one-element copy out of another array is read from there
        keys = []
        for kb in (key0, key1):
            w = writers.get(pid(kb), [])
            C = ops[w[0]] if len(w) == 1 else None
            if (C is not None and C.chain is not None and not C.chain.steps and kb.size == 1 and w[0] not in removed
                    and C.chain.first.buffer.dtype == kb.dtype):
                keys.append((C.chain.first.buffer, C.chain.first.offset))
                if uses[pid(kb)] == 1:
                    members.append(w[0])
                    kb._placeholder.elided = True
            else:
                keys.append((kb, 0))
        fused = Op(_label(*[ops[i] for i in sorted(members)]),
                   launch=K.threefry_stream(out, keys[0], keys[1], h, sources[0][1], sources[1][1], steps, n=count),
                   meta=('random_stream', out, 'halves', keys[0], keys[1], h, sources[0][1], sources[1][1], count, steps))
        fused.index = ops[last].index
        for b in [keys[0][0], keys[1][0]] + [st.operand.buffer for st in steps if st.operand is not None]:
            b.accesses.append(fused.index)
        for b in (x0, x1, aa, ab) + ((AC,) if chain_pos is not None else ()):
            b._placeholder.elided = True
        removed |= set(members)
        replacement[last] = fused
        if any(odd):
            sources[0][3]._placeholder.elided = True
            part    = next(ops[i].meta[2] for i in sources[0][2] if ops[i].meta[2].size != 1)
            sources = [(None, 0, writers[pid(part)][0], part)]
        #an iota nobody reads any more goes too
        for _, _, si, S in sources:
            uses[pid(S)] -= 1
            if uses[pid(S)] == 0 and si not in removed:
                removed.add(si)
                S._placeholder.elided = True
    return [replacement.get(i, op) for i, op in enumerate(ops) if i not in removed or i in replacement]


def _is_small(op) -> bool:
    '''An element-wise chain or a plain float column sum of a few workgroups, of a kind that has a batch kernel.'''
    if op.chain is None and not (op.conv is None and op.launch.kernel in K.REDUCE_BATCH_KERNELS + K.UPDATE_BATCH_KERNELS):
        return False
    if op.launch.kernel in K.TRANSPOSE_BATCH_KERNELS:
        #a tiled copy that swaps two dimensions (a network's kernels, transposed for its backward pass): batched up to a
        #larger size, a launch of a few microseconds carries little more than its own latency
        return op.launch.grid[0] * op.launch.grid[1] * op.launch.grid[2] <= K.TRANSPOSE_BATCH_MAX_BLOCKS
    return op.launch.kernel in K.BATCH_KERNELS and op.launch.grid[0] <= K.BATCH_MAX_BLOCKS


def _small_reads(op) -> tp.List:
    return _reads(op) if op.chain is not None else [b for b, _ in op.launch.buffers[1:]]


def _small_out(op):
    return op.chain.out if op.chain is not None else op.launch.buffers[0][0]


def _may_write(op) -> tp.List:
    '''Buffers an op may change: its result where the op's structure is known, else everything it touches.'''
    if op.chain is not None or op.conv is not None or (op.meta is not None and op.meta[0] in ('iota', 'concat_part', 'threefry', 'random_stream', 'reduce', 'update', 'window_sum', 'relu_backward', 'softmax', 'rows', 'conv_pack')):
        return _writes(op)
    return [b for b, _ in op.launch.buffers if b is not None]


def _written(op) -> tp.List:
    '''Buffers an op changes, by its launch's own record where its structure is not known otherwise.'''
    if op.chain is None and op.conv is None and op.meta is None:
        return [op.launch.buffers[k][0] for k in op.launch.written if op.launch.buffers[k][0] is not None]
    return _may_write(op)


def _touched(op) -> tp.List:
    if op.chain is not None or op.conv is not None:
        return _reads(op) + _writes(op)
    return [b for b, _ in op.launch.buffers if b is not None]


PACK_BATCH_ELEMENTS = 1 << 22          #weights that are packed by one launch, at least (16 MB)


def batch_packs(ops):
    '''Kernel operands that are packed for the matrix cores and depend on nothing the program computes (its weights) are
    packed several layers at a time, in front of the first of those layers: one launch per 16 MB of weights instead of one
    per layer, and not one for all of them, so that the first layers do not wait for weights of the last ones that are
    still being uploaded.'''
    from .ops import Op
    if not any(op.meta is not None and op.meta[0] == 'conv_pack' for op in ops):
        return ops
    written = set()
    for op in ops:
        written |= {id(b._placeholder) for b in _may_write(op)}
    result, group, size, at = [], [], 0, None
    def close():
        if len(group) > 1:
            batch = Op(_label(*group), launch=K.batch_launch([op.launch for op in group]))
            batch.index = group[0].index
            for op in group:
                for b, _ in op.launch.buffers:
                    b.accesses.append(batch.index)
            result[at] = batch
        group.clear()
    for op in ops:
        if op.meta is None or op.meta[0] != 'conv_pack' or id(op.meta[2].buffer._placeholder) in written:
            result.append(op)
            continue
        if not group:
            at, size = len(result), 0
            result.append(op)
        group.append(op)
        size += op.meta[3].K * op.meta[3].N
        if size >= PACK_BATCH_ELEMENTS:
            close()
    close()
    return result


#launches a program must save before its small chains are moved and batched. Replays of training steps, not batched and batched: two
#dense layers over 1000 rows, which save three, 78.4 and 69.0 us; programs that would save two, and are left as they are: two dense layers
#over 200 rows 61.5, 57.2, over 128 rows 55.8, 52.1, two convolutions on four images 88.0, 82.2, three dense layers over 61 rows 75.2, 72.5
BATCH_MIN_GAIN = 3


def batch_small_chains(ops):
    '''Programs with many little vectors (per-channel statistics, parameter updates of a training step)
    spend most of their launches on element-wise chains of a few workgroups, each paying a full launch
    latency. This pass

    1. moves every such chain that depends only on program inputs (or on chains moved before it) to the
       front, and every one whose result nothing but other moved chains reads to the end,
    2. sorts each run of consecutive small chains into dependency levels (read-after-write, write-after-read
       and write-after-write on the buffers) and turns every level's chains of one kernel variant into ONE
       launch of ew_chain_batch_* / reduce_cols_fsum_batch_*, and
    3. rebuilds the buffers' access positions from the final order, since storage is shared between
       buffers by those positions.

    Every chain computes what it computed before; only the order of independent launches changes.'''
    from .ops import Op
    pid = lambda b: id(b._placeholder)
    small = [_is_small(op) for op in ops]
    if sum(small) < BATCH_MIN_GAIN + 1:
        return ops

    # 1a. to the front
    written, touched, front = set(), set(), set()
    for i, op in enumerate(ops):
        if small[i] and not any(pid(b) in written for b in _small_reads(op)) and pid(_small_out(op)) not in touched:
            front.add(i)
            continue
        written |= {pid(b) for b in _may_write(op)}
        touched |= {pid(b) for b in _touched(op)}
    # 1b. to the end
    written, touched, back = set(), set(), set()
    for i in reversed(range(len(ops))):
        op = ops[i]
        if i not in front and small[i] and pid(_small_out(op)) not in touched and not any(pid(b) in written for b in _small_reads(op)):
            back.add(i)
            continue
        written |= {pid(b) for b in _may_write(op)}
        touched |= {pid(b) for b in _touched(op)}
    order = ([i for i in range(len(ops)) if i in front] + [i for i in range(len(ops)) if i not in front and i not in back]
             + [i for i in range(len(ops)) if i in back])
    moved = [ops[i] for i in order]

    # 2. runs of small chains -> levels -> batches
    result, saved, i = [], 0, 0
    while i < len(moved):
        if not _is_small(moved[i]):
            result.append(moved[i])
            i += 1
            continue
        j = i
        while j < len(moved) and j - i < 256 and _is_small(moved[j]):      #(levels are found pair by pair: bounded runs)
            j += 1
        run, level = moved[i:j], []
        for k, op in enumerate(run):
            reads, out = {pid(b) for b in _small_reads(op)}, pid(_small_out(op))
            lv = 0
            for q in range(k):
                q_reads, q_out = {pid(b) for b in _small_reads(run[q])}, pid(_small_out(run[q]))
                if q_out in reads or q_out == out or out in q_reads:
                    lv = max(lv, level[q] + 1)
            level.append(lv)
        for lv in range(max(level) + 1):
            by_kernel: tp.Dict[str, list] = {}
            for k, op in enumerate(run):
                if level[k] == lv:
                    by_kernel.setdefault(K.BATCH_KERNELS[op.launch.kernel], []).append(op)
            for group in by_kernel.values():
                if len(group) == 1:
                    result.append(group[0])
                    continue
                batch = Op(_label(*group), launch=K.batch_launch([op.launch for op in group]))
                batch.index = min(op.index for op in group)
                result.append(batch)
                saved += len(group) - 1
        i = j
    if saved < BATCH_MIN_GAIN:
        return ops

    # 3. access positions of every buffer in the order the launches now have
    fresh: tp.Dict[int, tp.Tuple[list, list]] = {}
    for position, op in enumerate(result):
        launches = op.launch.members or (op.launch,)
        for launch in launches:
            for b, _ in launch.buffers:
                if b is not None:
                    fresh.setdefault(id(b.accesses), (b.accesses, []))[1].append(position)
        op.index = position
    for accesses, positions in fresh.values():
        accesses[:] = positions
    return result
