'''Launch descriptors for the gfx950 kernels.

Where the reference turned an op into SPIR-V by pasting shapes into GLSL text and compiling it
at run time (vkjax/shaders.py:16-42, vkjax/ops.py:36-41), the kernels here are built ahead of
time and take shapes and strides as kernel arguments. Each function below lays out the argument
block of one kernel (a struct of 32-bit fields that follows the pointer arguments, mirroring the
`struct ...Params` in vkjax_amd/csrc/kernels/*.hip) and picks grid, block and kernel variant.
'''
import contextlib
import os
import re
import typing as tp

import numpy as np

from .buffers import Buffer

_KDIR = os.path.join(os.path.dirname(os.path.abspath(__file__)), 'csrc', 'kernels')


def _read_opcodes() -> tp.Dict[str, int]:
    text = open(os.path.join(_KDIR, 'ew_opcodes.h')).read()
    return {m.group(1): int(m.group(2)) for m in re.finditer(r'^EW_OP\((\w+),\s*(\d+)\)', text, re.M)}


EW = _read_opcodes()
EW_MAX_STEPS = 8
CONV_MAX_EPI = 6
BLOCK = 256


class _Choices:
    '''Which kernel variant a lowering picks where several would do. Every field has the value the heuristics work
    with; `overrides(...)` pins some of them for the duration of a `with` block, which is how tests reach every
    variant whatever the heuristics would choose, and how measurements compare variants.'''
    DEFAULTS = dict(
        ew_affine=None,                  #the straight-line affine kernel: None = where it pays, True = wherever it applies, False = never
        conv_tile=None,                  #name of the tile shape (CONV_TILES) instead of the estimate's choice
        conv_bk=None,                    #k step
        conv_chunk=None,                 #consecutive M tiles a lean block walks
        conv_blocks_per_cu=5,            #blocks of the lean 64 x 64 kernels a CU holds at once (94 registers); 0 = no evenly split grids
        conv_even_split_min_tiles=4.5,   #tiles per block from which an evenly split grid is used
        conv_general=False,              #never pick the lean kernel variant
        conv_b_general=False,            #element-wise loads of the kernel operand also where 16-byte loads would do
        conv_ksplit=None,                #the four-waves-per-tile kernel: always (where it applies) / never
        pool_gradient_2d=None,           #the 2-D kernels of a pooling gradient: None = where they apply, False = never, 'elements' = never the one for groups of 2 x 2 elements
        scatter_bucket_cap=None,         #slots per row in the sorted scatter-add's table of fixed-capacity buckets (0: no table)
        conv_dense_rows=None,            #the kernel for at most 16 output features: None = where it applies, False = never
        conv_mix=None,                   #mixed 64 x 64 / 32 x 32 tiling: None = by the heuristic, False = never, an int = that many M tiles stay 64 x 64
        conv_stem=None,                  #the kernels for images of very few features: None = where they pay, True = wherever they apply, 64 = with tiles of 64 positions, False = never
        conv_split=None,                 #the kernels on the bf16 matrix cores: None = where they pay, False = never, True or a tile's name = wherever they apply
        conv_split_slices=None,          #blocks that share a tile behind the whole rounds (None: by the estimate)
        conv_patch=None,                 #the bf16 kernels that hold a patch of the input in LDS: None = wherever they pay (a pinned conv_split: never), True = wherever they apply, 'fine' = wherever they apply, with their two sums, False = never
        conv_ragged=None,                #the bf16 kernel for 3 x 3 windows over any number of features: None = where it pays (a pinned conv_split: never), True = wherever no other patch kernel applies, False = never
        conv_short=None,                 #the bf16 kernels for dense rows of at most 64 features: None = where they pay (a pinned conv_split: never), True = wherever they apply, False = never
        wgrad_split=None,                #kernel gradients on the bf16 matrix cores: None = where they pay, False = never, a tile's name = wherever it applies
        wgrad_slices=None,               #slices of a kernel gradient's contraction (None: by the estimate)
        conv_k_splits=None,              #slices a contraction is cut into where that applies (None: by the heuristic, 1: never)
        conv_shares=None,                #blocks that share a tile of the four-waves-per-tile kernels and add its slices themselves (None: by the estimate; a pinned conv_k_splits or conv_split: never, 1: never)
        conv_xcd_columns='ranges',       #four-waves-per-tile kernels: how tiles go to the XCDs ('ranges': row by row or column by column, by the operands' sizes; 0: row by row, 'columns': column by column, a number or None: rectangles of tiles)
        scatter_sort_threshold=1 << 18,  #update elements from which a row scatter-add sorts its updates instead of using atomics
        scatter_short_rows=None,         #several table rows per wave in the sorted scatter-add: None = where it pays, True = wherever rows are short enough, False = never
        reuse_equal_equations=True,      #an equation that repeats an earlier one is bound to that one's buffer
    )

    def __init__(self):
        self.__dict__.update(self.DEFAULTS)


CHOICES = _Choices()


@contextlib.contextmanager
def overrides(**pinned):
    '''`with overrides(conv_tile='64x64', conv_bk=32): ...` - programs built inside the block use the given
    choices (fields of `_Choices.DEFAULTS`); the previous values return when the block is left.'''
    unknown = set(pinned) - set(_Choices.DEFAULTS)
    if unknown:
        raise TypeError(f'overrides: unknown choice(s) {sorted(unknown)}; known: {sorted(_Choices.DEFAULTS)}')
    saved = {name: getattr(CHOICES, name) for name in pinned}
    CHOICES.__dict__.update(pinned)
    try:
        yield CHOICES
    finally:
        CHOICES.__dict__.update(saved)


class Launch(tp.NamedTuple):
    kernel:  str
    grid:    tp.Tuple[int, int, int]
    block:   tp.Tuple[int, int, int]
    buffers: tp.List[tp.Tuple[tp.Optional[Buffer], int]]     #(buffer, byte offset) in argument order
    params:  bytes
    lds:     int = 0
    #algorithmic work of this launch, for roofline accounting
    bytes_moved: int = 0
    flops:       int = 0
    #a batch launch: the launches it evaluates, described to the kernel by a table in device memory
    #that is written when the launch is recorded (it holds device addresses)
    members: tp.Tuple['Launch', ...] = ()
    #the kernel stores its result (its first array) past the caches when bit 31 of its first parameter word is set
    #(see with_streamed_result)
    streamable: bool = False
    #which of `buffers` the kernel writes (positions); everything else it only reads
    written: tp.Tuple[int, ...] = (0,)
    #which of `buffers` are scratch that other launches use too and that holds nothing (counters: zeros) between launches
    scratch: tp.Tuple[int, ...] = ()


def _u32(*values) -> bytes:
    return np.asarray([int(v) & 0xFFFFFFFF for v in values], dtype=np.uint32).tobytes()


def _i32(*values) -> bytes:
    return np.asarray([int(v) for v in values], dtype=np.int32).tobytes()


def _pad(seq, n, fill=0):
    seq = list(seq)
    assert len(seq) <= n, (seq, n)
    return seq + [fill] * (n - len(seq))


def _cdiv(a, b):
    return -(-int(a) // int(b))


def row_major_strides(shape) -> tp.Tuple[int, ...]:
    strides, acc = [], 1
    for s in reversed(shape):
        strides.append(acc)
        acc *= int(s)
    return tuple(reversed(strides))


# --------------------------------------------------------------------------- element-wise chains

class EwOperand(tp.NamedTuple):
    '''An array read by an element-wise chain: element `coords` of the output reads
    buffer[offset + sum(coords * strides)] (strides in elements, one per output dim).'''
    buffer:  Buffer
    offset:  int
    strides: tp.Tuple[int, ...]


class EwStep(tp.NamedTuple):
    op:           int
    operand:      tp.Optional[EwOperand] = None
    operand_left: bool = False
    imm:          int = 0


class EwChain:
    '''out = step_n(... step_1(first) ...) over `shape`.'''
    def __init__(self, out: Buffer, shape, first: EwOperand, steps: tp.Sequence[EwStep]):
        self.out, self.shape, self.first, self.steps = out, tuple(int(s) for s in shape), first, list(steps)

    def operands(self) -> tp.List[tp.Optional[EwOperand]]:
        return [self.first] + [s.operand for s in self.steps]


def broadcast_operand(buf: Buffer, out_shape) -> EwOperand:
    '''Trailing-aligned numpy-style broadcast of `buf` to `out_shape` (reference: vkjax/ops.py:160-184).'''
    out_shape = tuple(out_shape)
    in_shape  = tuple(buf.shape)
    if len(in_shape) > len(out_shape):
        raise ValueError(f'Cannot broadcast from {in_shape} to {out_shape}')
    in_strides = row_major_strides(in_shape)
    strides    = [0] * len(out_shape)
    for i in range(1, len(in_shape) + 1):
        old, new = in_shape[-i], out_shape[-i]
        if old != new and old != 1:
            raise ValueError(f'Cannot broadcast from {in_shape} to {out_shape}')
        strides[-i] = in_strides[-i] if old == new and old != 1 else 0
    return EwOperand(buf, 0, tuple(strides))


def _collapse(shape, stride_sets):
    '''Drop size-1 dims and merge neighbours that every operand walks contiguously.'''
    dims    = [(s, [st[i] for st in stride_sets]) for i, s in enumerate(shape) if s != 1]
    if not dims:
        return [1], [[0] for _ in stride_sets]
    merged = [dims[0]]
    for size, strides in dims[1:]:
        psize, pstrides = merged[-1]
        if all(ps == s * size for ps, s in zip(pstrides, strides)):
            merged[-1] = (psize * size, strides)
        else:
            merged.append((size, strides))
    out_dims    = [m[0] for m in merged]
    out_strides = [[m[1][k] for m in merged] for k in range(len(stride_sets))]
    return out_dims, out_strides


def lower_ew_chain(chain: EwChain) -> Launch:
    operands = chain.operands()
    nsteps   = len(operands)
    if nsteps > EW_MAX_STEPS:
        raise ValueError(f'element-wise chain of {nsteps} steps exceeds the kernel limit of {EW_MAX_STEPS}')
    n = int(np.prod(chain.shape, dtype=np.int64))
    present = [o for o in operands if o is not None]
    #the output is walked contiguously; include its strides so that merging respects it
    out_strides = row_major_strides(chain.shape)
    dims, strides = _collapse(chain.shape, [out_strides] + [o.strides for o in present])
    if len(dims) > 4:
        raise NotImplementedError(f'element-wise access pattern with {len(dims)} irreducible dimensions: {chain.shape}')
    ndim    = len(dims)
    strides = strides[1:]
    transposed = _as_tiled_transpose(chain, dims, strides)
    if transposed is not None:
        return transposed
    affine = _as_affine_chain(chain, n, dims, strides)
    if affine is not None:
        return affine
    vec = 4
    if n % 4 or dims[-1] % 4:
        vec = 1
    for o, st in zip(present, strides):
        if st[-1] not in (0, 1):
            vec = 1
        elif st[-1] == 1 and (o.offset % 4 or any(s % 4 for s in st[:-1])):
            vec = 1
    magics = [_magic_division(d) for d in _pad(dims, 4, 1)]
    ops, flags, imms, stride_rows, buffers, extents, bases = [], [], [], [], [], [], []
    it = iter(strides)
    for k, o in enumerate(operands):
        step = chain.steps[k - 1] if k > 0 else None
        ops.append(step.op if step else 0)
        imms.append(step.imm if step else 0)
        flag = 2 if (step and step.operand_left) else 0
        if o is None:
            stride_rows.append([0, 0, 0, 0])
            buffers.append((None, 0))
            extents.append(0)
            bases.append(0)
        else:
            st = next(it)
            if o.buffer.size * 4 >= 2**32:
                raise NotImplementedError('element-wise operand of 4 GiB or more')
            extents.append(o.buffer.size * 4)
            bases.append(o.offset)
            flag |= 1 | (4 if st[-1] == 1 else 0)
            #simple addressing patterns the kernel resolves without multiplications
            if all(s == 0 for s in st):
                flag |= 3 << 4 | 64
            elif tuple(st) == row_major_strides(dims):
                flag |= 1 << 4
            elif st[-1] == 1 and all(s == 0 for s in st[:-1]):
                flag |= 2 << 4
                #a thread's vectors are BLOCK * vec elements apart: the same coordinate when the dimension's length divides that
                if (BLOCK * vec) % dims[-1] == 0:
                    flag |= 64
            stride_rows.append(_pad(st, 4))
            buffers.append((o.buffer, 0))
        flags.append(flag)
    while len(stride_rows) < EW_MAX_STEPS:
        stride_rows.append([0, 0, 0, 0])
        buffers.append((None, 0))
    params = (_u32(n, ndim, *_pad(dims, 4, 1), nsteps, *_pad(ops, EW_MAX_STEPS), *_pad(flags, EW_MAX_STEPS),
                   *_pad(imms, EW_MAX_STEPS))
              + _i32(*[s for row in stride_rows for s in row]) + _u32(*_pad(extents, EW_MAX_STEPS), *_pad(bases, EW_MAX_STEPS))
              + _u32(*[m for m, _ in magics], *[sh for _, sh in magics]))
    nbytes = 4 * n + sum(4 * min(n, o.buffer.size) for o in present)
    if n >= 2**31:
        raise NotImplementedError(f'element-wise op over {n} elements exceeds 32-bit indexing')
    slots = 2 if nsteps <= 2 else 4 if nsteps <= 4 else 6 if nsteps <= 6 else 8
    per_thread = {2: 1, 4: 2, 6: 2, 8: 1}[slots]               #vectors a thread works on (the kernel's U)
    return Launch(f'ew_chain_v{vec}_s{slots}', (_cdiv(_cdiv(n, vec), BLOCK * per_thread), 1, 1), (BLOCK, 1, 1),
                  [(chain.out, 0)] + buffers, params, bytes_moved=nbytes, streamable=vec == 4)


EW_AFFINE_BIG_ELEMENTS = 1 << 22
#Results from this size on that no later launch of the program reads are stored with the nontemporal hint: such an array
#only pushes out of the caches what could be reused, and the stores of a launch that reads and writes run faster past the
#L2 (relu on 64 M elements 92 -> 76 us, exp 96 -> 81 us). Results that the next launch reads are left to the caches.
STREAM_RESULT_MIN_BYTES = 64 << 20
STREAM_RESULT_BIT = 1 << 31
#kernels that add to what their result array already holds (their first array is read as well as written)
ACCUMULATING_KERNELS = ('scatter_add_rows', 'scatter_add_general')


def with_streamed_result(launch: Launch) -> Launch:
    '''`launch` with the flag set that makes its kernel store the result past the caches (bit 31 of the first
    parameter word, an element count below 2**31 in every kernel that is marked streamable).'''
    assert launch.streamable and not launch.members
    first = int(np.frombuffer(launch.params[:4], np.uint32)[0])
    assert first < STREAM_RESULT_BIT
    return launch._replace(params=_u32(first | STREAM_RESULT_BIT) + launch.params[4:])


def _as_affine_chain(chain: EwChain, n: int, dims, strides) -> tp.Optional[Launch]:
    '''ew_affine_v4 for float chains of the form ((first + s1 + s2 + s3) - vsub) * vmul + vadd + full, max(., floor)
    (every part optional, in this order; s and full arrays of the output's shape, v vectors over the fastest
    dimension, floor one value), for chains of more than four operands: a small launch is mostly the interpreter's
    latency, and on large arrays the interpreter's instructions cost a fifth of the bandwidth (batch norm + ReLU on
    51 M elements 4.5 TB/s, here 5.7). Shorter chains keep the general kernel, which is as fast for them and whose
    small launches are batched with their neighbours.'''
    operands = chain.operands()
    if (CHOICES.ew_affine is False or not chain.steps or any(o is None for o in operands) or n % 4 or dims[-1] % 4 or n * 4 >= 2**32 - 2**16
            or len(dims) > 2 or (CHOICES.ew_affine is None and len(operands) <= 4)
            or any(np.dtype(b.dtype) != np.float32 for b in [chain.out] + [o.buffer for o in operands])):
        return None
    dense = row_major_strides(dims)
    kind  = lambda st: ('full' if tuple(st) == dense else 'vec' if len(dims) == 2 and tuple(st) == (0, 1)
                        else 'one' if all(s == 0 for s in st) else None)
    kinds = [kind(st) for st in strides]
    if kinds[0] != 'full' or (len(dims) == 1 and 'vec' in kinds):
        return None
    steps, k = list(zip(chain.steps, operands[1:], kinds[1:])), 0
    sums, slot = [], {}
    while k < len(steps) and len(sums) < 3 and steps[k][0].op == EW['ADD_F'] and steps[k][2] == 'full':
        sums.append(steps[k][1]); k += 1
    template = ((0, EW['SUB_F'], 'vec', False), (1, EW['MUL_F'], 'vec', None), (2, EW['ADD_F'], 'vec', None),
                (3, EW['ADD_F'], 'full', None), (4, EW['MAX_F'], 'one', False))
    t = 0
    while k < len(steps):
        step, operand, what = steps[k]
        while t < len(template) and not (step.op == template[t][1] and what == template[t][2]
                                         and (template[t][3] is None or bool(step.operand_left) == template[t][3])):
            t += 1
        if t == len(template):
            return None
        slot[template[t][0]] = operand
        t += 1; k += 1
    if not sums and not slot:
        return None
    C = dims[-1] if len(dims) == 2 else 4
    if any(o.buffer.size != C for b, o in slot.items() if b in (0, 1, 2)):
        return None
    magic, shift = _magic_division(C // 4)
    at = lambda o: (o.buffer, o.offset * 4) if o is not None else (None, 0)
    buffers = ([(chain.out, 0), at(operands[0])] + [at(o) for o in _pad(sums, 3, None)]
               + [at(slot.get(b)) for b in range(5)])
    params  = _u32(n, C // 4, magic, shift, len(sums), sum(1 << b for b in slot))
    nbytes  = 4 * n + sum(4 * min(n, o.buffer.size) for o in operands)
    #(arrays of more than 16 MB: the variant that skips absent operands instead of loading through empty descriptors)
    kernel = 'ew_affine_big_v4' if n > EW_AFFINE_BIG_ELEMENTS else 'ew_affine_v4'
    return Launch(kernel, (_cdiv(n // 4, 2 * BLOCK), 1, 1), (BLOCK, 1, 1), buffers, params, bytes_moved=nbytes, streamable=True)


EW_BATCH_KERNELS     = ('ew_chain_v1_s2', 'ew_chain_v1_s4', 'ew_chain_v4_s2', 'ew_chain_v4_s4')
REDUCE_BATCH_KERNELS = ('reduce_cols_fsum_v1', 'reduce_cols_fsum_v4')
UPDATE_BATCH_KERNELS = ('reduce_cols_fsum_update_v1', 'reduce_cols_fsum_update_v4')
TRANSPOSE_BATCH_KERNELS = ('transpose_tiled_v4', 'transpose_tiled_v4_t128')
BATCH_KERNELS        = {**{k: k.replace('ew_chain_', 'ew_chain_batch_') for k in EW_BATCH_KERNELS},
                        **{k: k.replace('fsum_', 'fsum_batch_') for k in REDUCE_BATCH_KERNELS},
                        **{k: 'reduce_cols_fsum_batch_update' for k in UPDATE_BATCH_KERNELS},
                        **{k: k.replace('tiled_', 'tiled_batch_') for k in TRANSPOSE_BATCH_KERNELS},
                        'conv_split_pack': 'conv_split_pack_layers'}
EW_BATCH_ENTRY_BYTES        = 432
REDUCE_BATCH_ENTRY_BYTES    = 56
TRANSPOSE_BATCH_ENTRY_BYTES = 48
PACK_BATCH_ENTRY_BYTES      = 56
BATCH_MAX_BLOCKS         = 4096        #launches of more workgroups than this keep a launch of their own
#column sums of up to a workgroup per CU trade the width of a block for more blocks. Sums of R rows alone, at 16 and at 256
#workgroups: 937 x 1728 7.0, 3.8 us; 256 x 4096 4.6, 2.8; 2000 x 4096 23.4, 6.6; 128 x 9408 3.5, 2.7; 937 x 30000 25.1, 19.1; at 512
#workgroups 937 x 9408 takes 6.1 instead of 8.3 and 937 x 30000 20.7
REDUCE_NARROW_MAX_BLOCKS = 256
TRANSPOSE_BATCH_MAX_BLOCKS = 1024      #... tiled transposes (the kernels of a network, for its backward pass) up to this many


def _blocks(launch: Launch) -> int:
    return launch.grid[0] * launch.grid[1] * launch.grid[2]


def batch_launch(members: tp.Sequence[Launch]) -> Launch:
    '''One launch for several small launches of one batch kernel (element-wise chains or float column sums)
    that do not depend on one another.'''
    kernel = BATCH_KERNELS[members[0].kernel]
    assert all(BATCH_KERNELS[m.kernel] == kernel and not m.members for m in members), [m.kernel for m in members]
    return Launch(kernel, (sum(_blocks(m) for m in members), 1, 1), (BLOCK, 1, 1), [],
                  _u32(len(members)), bytes_moved=sum(m.bytes_moved for m in members), members=tuple(members))


def batch_table(launch: Launch, device_address: tp.Callable[[Buffer], int]) -> np.ndarray:
    '''The table of a batch launch as uint32 words, one entry per member: {first workgroup, 0 (tiled transposes: the
    x extent of the member's grid), the addresses of the member's arrays (0 = none), the member's parameter block
    (tiled transposes: then the y extent of its grid)}, padded to a multiple of 8 bytes.'''
    kind = launch.members[0].kernel
    is_chain, is_transpose = kind in EW_BATCH_KERNELS, kind in TRANSPOSE_BATCH_KERNELS
    entry_bytes, pointers = ((EW_BATCH_ENTRY_BYTES, 1 + EW_MAX_STEPS) if is_chain else
                             (TRANSPOSE_BATCH_ENTRY_BYTES, 2) if is_transpose else
                             (PACK_BATCH_ENTRY_BYTES, 2) if kind == 'conv_split_pack' else (REDUCE_BATCH_ENTRY_BYTES, 4 if kind in UPDATE_BATCH_KERNELS else 2))
    rows, first = [], 0
    for m in launch.members:
        assert len(m.buffers) == pointers, (m.kernel, len(m.buffers))
        addresses = [device_address(b) + off if b is not None else 0 for b, off in m.buffers]
        #(a transpose has a three-dimensional grid of its own: its x extent follows first_block, its y extent the parameters)
        row = (_u32(first, m.grid[0] if is_transpose else 0) + np.asarray(addresses, dtype=np.uint64).tobytes() + m.params
               + (_u32(m.grid[1]) if is_transpose else b''))
        rows.append(row + bytes(entry_bytes - len(row)))
        first += _blocks(m)
    table = b''.join(rows)
    assert len(table) == entry_bytes * len(launch.members)
    return np.frombuffer(table, dtype=np.uint32).copy()


TRANSPOSE_BIG_TILES = True


def _as_tiled_transpose(chain: EwChain, dims, strides) -> tp.Optional[Launch]:
    '''A pure copy whose collapsed form is out[b, i, j] = in[b * sb + j * sj + i] (the two fastest dimensions
    trade places) goes through the LDS-tiled kernel when both of them are at least 16 long.'''
    if chain.steps or len(dims) not in (2, 3):
        return None
    st = strides[0]
    B, I, J = ([1] + list(dims))[-3:]
    sb = st[0] if len(dims) == 3 else 0
    if st[-2] != 1 or st[-1] < I or I < 16 or J < 16 or B > 65535 or _cdiv(I, 64) > 65535:
        return None
    src = chain.first
    if src.buffer.size * 4 >= 2**32:
        return None
    n = B * I * J
    vec = all(v % 4 == 0 for v in (I, J, st[-1], sb, src.offset))
    if vec and I >= 128 and J >= 128 and I * J >= 1 << 16 and TRANSPOSE_BIG_TILES:
        return Launch('transpose_tiled_v4_t128', (_cdiv(J, 128), _cdiv(I, 128), B), (BLOCK, 1, 1), [(chain.out, 0), (src.buffer, src.offset * 4)],
                      _u32(B, I, J, sb, st[-1]), lds=0, bytes_moved=8 * n, streamable=True)
    return Launch('transpose_tiled_v4' if vec else 'transpose_tiled', (_cdiv(J, 64), _cdiv(I, 64), B), (BLOCK, 1, 1), [(chain.out, 0), (src.buffer, src.offset * 4)],
                  _u32(B, I, J, sb, st[-1]), bytes_moved=8 * n, streamable=bool(vec))


def iota(out: Buffer, dimension: int) -> Launch:
    n     = out.size
    inner = int(np.prod(out.shape[dimension + 1:], dtype=np.int64))
    size  = out.shape[dimension]
    vec   = 4 if n % 4 == 0 else 1
    return Launch(f'iota_nd_v{vec}', (_cdiv(_cdiv(n, vec), BLOCK), 1, 1), (BLOCK, 1, 1), [(out, 0)],
                  _u32(n, inner, size, int(out.dtype == np.float32)), bytes_moved=4 * n)


def fill(out: Buffer, word: int) -> Launch:
    n = out.size
    return Launch('fill_u32', (_cdiv(_cdiv(n, 4), BLOCK), 1, 1), (BLOCK, 1, 1), [(out, 0)], _u32(n, word), bytes_moved=4 * n)


def concat_part(out: Buffer, part: Buffer, dimension: int, offset_along_dim: int) -> Launch:
    inner      = int(np.prod(out.shape[dimension + 1:], dtype=np.int64))
    part_inner = part.shape[dimension] * inner
    out_inner  = out.shape[dimension] * inner
    n   = part.size
    vec = 4 if (part_inner % 4 == 0 and out_inner % 4 == 0 and (offset_along_dim * inner) % 4 == 0) else 1
    return Launch(f'concat_part_v{vec}', (_cdiv(_cdiv(n, vec), BLOCK), 1, 1), (BLOCK, 1, 1), [(out, 0), (part, 0)],
                  _u32(n, part_inner, out_inner, offset_along_dim * inner), bytes_moved=8 * n, streamable=vec == 4 and n < 2**31)


TF_MAX_STEPS = 8


_UNIFORM_CHAIN_OPS = [EW[name] for name in ('SHR_L', 'OR_X', 'SUB_F', 'MUL_F', 'ADD_F', 'MAX_F')]


class KeySplit(tp.NamedTuple):
    '''Two words of what a stream without steps would store: its layout (halves or pairs), blocks, counters and size.'''
    layout: str
    h:      int
    c0:     int
    c1:     int
    n:      int
    words:  tp.Tuple[int, int]


#blocks of a launch that splits its key itself: eight per CU, every thread on several vectors
KEY_SPLIT_BLOCKS = 2048


def threefry_stream(out: Buffer, key0: tp.Tuple[Buffer, int], key1: tp.Tuple[Buffer, int], h: int, c0: int, c1: int,
                    steps: tp.Sequence[EwStep], layout: str = 'halves', n: tp.Optional[int] = None,
                    key_split: tp.Optional[KeySplit] = None) -> Launch:
    '''Random words from counters generated in registers, the element-wise `steps` (operands: single
    values) applied before the only store. `h` blocks are run; the key words are given as
    (buffer, element offset). Layouts:
      halves  out[j], out[h + j] = steps(threefry2x32(key, c0 + j, c1 + j)); `n` (2h or 2h - 1) is the
              number of elements stored, and with n == 2h - 1 the last x1 counter is 0
      xor     out[j] = steps(y0 ^ y1) with y = threefry2x32(key, c0, c1 + j)
      pairs   out[2j], out[2j + 1] = threefry2x32(key, c0, c1 + j)  (no steps)
    `key_split`: key0 and key1 are the key that was split, and the key words two words of that split.'''
    if len(steps) > TF_MAX_STEPS:
        raise ValueError('too many steps')
    if layout == 'pairs' and steps:
        raise ValueError('the pairs layout takes no steps')
    n = 2 * h if n is None else n
    assert layout != 'halves' or n in (2 * h, 2 * h - 1)
    flags, buffers = [], []
    for s in steps:
        if s.operand is not None:
            assert s.operand.buffer.size == 1 and s.operand.offset == 0
        flags.append((1 if s.operand is not None else 0) | (2 if s.operand_left else 0))
        buffers.append((s.operand.buffer if s.operand is not None else None, 0))
    vec = 4 if h % 4 == 0 and (n == 2 * h if layout == 'halves' else layout == 'xor') else 1
    params = _u32(h, c0, c1, len(steps), *_pad([s.op for s in steps], TF_MAX_STEPS), *_pad(flags, TF_MAX_STEPS),
                  *_pad([s.imm for s in steps], TF_MAX_STEPS), n,
                  *(({'halves': 1, 'pairs': 3}[key_split.layout], *key_split[1:5], *key_split.words) if key_split else (0,) * 7))
    kernel = {'halves': 'threefry2x32_stream', 'xor': 'threefry2x32_stream_xor', 'pairs': 'threefry2x32_stream_pairs'}[layout]
    kernel += f'_v{vec}'
    #jax.random.uniform's chain has kernels of its own with the steps compiled in
    if [s.op for s in steps] == _UNIFORM_CHAIN_OPS and flags == [1, 1, 1, 1, 1, 3] and all(s.imm == 0 for s in steps) and layout != 'pairs':
        kernel = kernel.replace('_v4', '_uniform_v4') if vec == 4 else kernel + '_uniform'
    blocks = _cdiv(_cdiv(h, vec), BLOCK)
    if key_split and layout != 'pairs':
        blocks = min(blocks, KEY_SPLIT_BLOCKS)
    return Launch(kernel, (blocks, 1, 1), (BLOCK, 1, 1),
                  [(out, 0), (key0[0], key0[1] * 4), (key1[0], key1[1] * 4)] + _pad(buffers, TF_MAX_STEPS, (None, 0)), params,
                  bytes_moved=4 * (h if layout == 'xor' else n))


# --------------------------------------------------------------------------- conv / dot

class ConvGeometry(tp.NamedTuple):
    '''Implicit-GEMM view of a convolution or matrix product (see csrc/kernels/conv_gemm.hip).'''
    batch: int; Ho: int; Wo: int; N: int
    H: int; W: int; Cin: int; KH: int; KW: int
    SH: int = 1; SW: int = 1; PH: int = 0; PW: int = 0; DH: int = 1; DW: int = 1; LH: int = 1; LW: int = 1
    xs: tp.Tuple[int, int, int, int] = (0, 0, 0, 1)      #lhs strides: batch, y, x, feature
    ws: tp.Tuple[int, int, int, int] = (0, 0, 0, 1)      #rhs strides: ky, kx, in feature, out feature
    os: tp.Tuple[int, int, int, int] = (0, 0, 0, 1)      #out strides: batch, y, x, feature
    #> 1: the contraction is cut into this many slices, each summed by blocks of its own into its own [M, N] matrix of
    #the result array (no epilogue); another launch adds the slices
    k_splits: int = 1
    #how the kernels on the bf16 matrix cores share the product out, or None: the others compute it
    split: tp.Optional['ConvSplit'] = None
    #how blocks share the tiles of a four-waves-per-tile kernel, or None: one block per tile
    shares: tp.Optional['ConvShares'] = None

    @property
    def M(self): return self.batch * self.Ho * self.Wo
    @property
    def K(self): return self.KH * self.KW * self.Cin


class WgradGeometry(tp.NamedTuple):
    '''Kernel gradient of an NHWC / HWIO convolution in the forward convolution's own terms: X is
    [images, H, W, C], the output cotangent G is [images, Ho, Wo, N], the result [KH, KW, C, N]
    (see csrc/kernels/wgrad_gemm.hip). A product X^T G of row-major matrices is the 1x1 case.'''
    images: int; Ho: int; Wo: int; H: int; W: int; C: int; KH: int; KW: int; N: int
    SH: int = 1; SW: int = 1; PH: int = 0; PW: int = 0; DH: int = 1; DW: int = 1

    @property
    def pixels(self): return self.images * self.Ho * self.Wo
    @property
    def M(self): return self.KH * self.KW * self.C


def choose_wgrad_splits(g: WgradGeometry, compute_units: int = 256) -> int:
    '''Slices of the contraction: enough blocks to fill the chip several times over, at least four
    k steps of 32 pixels per slice.'''
    tiles = _cdiv(g.M, 64) * _cdiv(g.N, 64)
    want  = _cdiv(4 * compute_units, tiles)
    return max(1, min(want, g.pixels // 128, 1024))


#Tiles of the kernel gradients on the bf16 matrix cores (csrc/kernels/wgrad_split.h): (BM, BN, blocks a CU holds (one of 128 x 128: of
#two groups of four waves, the others have one), microseconds of such
#a CU per block and k tile of 32 pixels, measured on ResNet-50's layers at batch 64, loads of X it is built for: 16 bytes / words)
WGRAD_SPLIT_TILES = {'128x128': (128, 128, 1, 1.55, 'a'), '128x64': (128, 64, 3, 0.95, 'a'), '64x128': (64, 128, 3, 0.95, 'a'), '64x64': (64, 64, 4, 0.57, 'as')}
#Below this many operations the fp32 kernels are as fast: 2000 x 1024 x 512 (2.1 GFLOP) takes 28 us there and 22 here, 1000 x 784 x 300
#(0.5) 12.6 and 12.8, 3x3 on 4 x 14 x 14 x 256 (0.9) 18.4 and 18.8.
WGRAD_SPLIT_MIN_FLOPS = 1.5e9
WGRAD_SPLIT_MAX_SLICES = 1024


class WgradPlan(tp.NamedTuple):
    '''The tile of the kernel on the bf16 matrix cores, or None for the one on fp32 products; slices of the contraction.'''
    tile:   tp.Optional[str]
    splits: int


def _wgrad_loads(g: WgradGeometry) -> str:
    return ('a' if g.C % 4 == 0 else 's') + ('a' if g.N % 4 == 0 else 's')


def wgrad_split_applies(tile: str, g: WgradGeometry) -> bool:
    '''The kernels are built for G in 16-byte loads; a pixel's (y, x) and a tap's offset are added as 16-bit numbers, which
    the bounds keep from running over.'''
    if g.N % 4 != 0 or _wgrad_loads(g)[0] not in WGRAD_SPLIT_TILES[tile][4]:
        return False
    tap = lambda k, d, p: max(abs(p), abs((k - 1) * d - p))
    return _wgrad_flat(g) or (max(g.H, g.W) <= 0x2000 and max(tap(g.KH, g.DH, g.PH), tap(g.KW, g.DW, g.PW)) < 0x1000
                              and max((g.Ho - 1) * g.SH, (g.Wo - 1) * g.SW) < 0x3000)


def wgrad_plan(g: WgradGeometry, compute_units: int = 256) -> WgradPlan:
    '''The tile and the number of slices with the smallest estimated time: the k tiles of the CU with the most blocks (one alone on a
    CU takes 1.3 times as long as one of as many as it holds), four microseconds to start and store, and the partial results written and added at 8 TB/s (at 3,
    which takes a quarter fewer slices, ResNet-50's training step takes 12.87 instead of 12.71 ms; at 20 it is as fast).'''
    fp32 = WgradPlan(None, choose_wgrad_splits(g, compute_units))
    if (CHOICES.wgrad_split is False or (CHOICES.wgrad_split is None and 2 * g.pixels * g.M * g.N < WGRAD_SPLIT_MIN_FLOPS)):
        return fp32
    ktiles, best = _cdiv(g.pixels, 32), None
    for tile, (bm, bn, resident, step, _) in WGRAD_SPLIT_TILES.items():
        if CHOICES.wgrad_split not in (None, tile) or not wgrad_split_applies(tile, g):
            continue
        tiles = _cdiv(g.M, bm) * _cdiv(g.N, bn)
        if CHOICES.wgrad_slices is not None:
            counts = {min(ktiles, CHOICES.wgrad_slices)}
        else:                                         #those that fill a number of rounds of one block per CU
            counts = {max(1, min(r * compute_units // tiles, ktiles // 4, WGRAD_SPLIT_MAX_SLICES)) for r in range(1, 9)}
        for splits in sorted(counts):
            per    = _cdiv(ktiles, splits)
            splits = _cdiv(ktiles, per)
            each   = _cdiv(tiles * splits, compute_units)
            alone  = 0.3 * max(0, resident - each) / max(1, resident - 1)
            time   = each * per * step * (1 + alone) + 4 + (3 + splits * g.M * g.N * 8 / 8e6 if splits > 1 else 0)
            if best is None or time < best[0]:
                best = (time, WgradPlan(tile, splits))
    return best[1] if best else fp32


def _wgrad_flat(g: WgradGeometry) -> bool:
    '''Pixel p's features start at p * C: a product of matrices, or a 1 x 1 window at a stride of 1 without padding.'''
    return g.KH == g.KW == g.SH == g.SW == 1 and g.PH == g.PW == 0 and (g.H, g.W) == (g.Ho, g.Wo)


def wgrad_gemm(out: Buffer, x: Buffer, cot: Buffer, g: WgradGeometry, splits: int, tile: tp.Optional[str] = None) -> Launch:
    '''`out` holds `splits` partial results of M * N elements each (the result itself when splits == 1). `tile`: one of
    WGRAD_SPLIT_TILES, for the kernel on the bf16 matrix cores.'''
    for name, b in (('input', x), ('cotangent', cot)):
        if b.size * 4 >= 2**31:
            raise NotImplementedError(f'kernel gradient: {name} of {b.size * 4} bytes exceeds the 2 GiB the kernel addresses')
    assert x.size == g.images * g.H * g.W * g.C and cot.size == g.pixels * g.N and out.size == splits * g.M * g.N
    per_split = _cdiv(_cdiv(g.pixels, splits), 32) * 32
    assert per_split * splits >= g.pixels
    magics = [v for d in (g.Ho * g.Wo, g.Wo, g.C, g.KW) for v in _magic_division(d)]
    params = _i32(g.pixels, g.M, g.N, g.Ho, g.Wo, g.H, g.W, g.C, g.KW, g.SH, g.SW, g.PH, g.PW, g.DH, g.DW, per_split) \
           + _u32(*magics, x.size * 4, cot.size * 4)
    loads = _wgrad_loads(g)
    work  = dict(bytes_moved=4 * (x.size + cot.size + out.size), flops=2 * g.pixels * g.M * g.N)
    if tile is not None:
        bm, bn = WGRAD_SPLIT_TILES[tile][:2]
        tiles_m, tiles_n = _cdiv(g.M, bm), _cdiv(g.N, bn)
        return Launch(f'wgrad_split_{tile}_{loads}', (tiles_m * tiles_n * splits, 1, 1), (512 if tile == '128x128' else 256, 1, 1), [(out, 0), (x, 0), (cot, 0)],
                      params + _i32(tiles_m, tiles_n, _wgrad_flat(g)), **work)
    return Launch(f'wgrad_gemm_64x64_{loads}', (_cdiv(g.N, 64), _cdiv(g.M, 64), splits), (256, 1, 1), [(out, 0), (x, 0), (cot, 0)], params, **work)


class ConvDerivedOperand(tp.NamedTuple):
    '''A per-feature epilogue operand that the kernel computes instead of reading: `first` and the
    step operands are buffers of N values or of one value.'''
    first: Buffer
    steps: tp.Tuple[tp.Tuple[int, tp.Optional[Buffer], bool], ...]       #(opcode, operand or None, operand is the left argument)


class ConvEpilogueStep(tp.NamedTuple):
    op:           int
    kind:         int                    #1 scalar, 2 per-feature vector [N], 3 full tensor laid out like the output
    operand:      tp.Optional[Buffer]    #None when `derived` says how to compute it
    operand_left: bool = False
    derived:      tp.Optional[ConvDerivedOperand] = None
    bounds:       tp.Tuple[Buffer, ...] = ()


#A pseudo step: the value as it stands at this point of the epilogue is ALSO stored to `operand`, an array laid
#out like the result (the centred convolution result a backward pass needs besides the activation)
CONV_TAP = -1
#A pseudo step, the last of an epilogue: the rows of the result are replaced by their softmax before the store;
#`operand`, if not None, is an int32 array [M] that receives each row's arg-max. Only the kernel for products with at
#most 16 output features (dense_rows_n16) can do this.
CONV_SOFTMAX = -2


#A pseudo step: the value is kept where `operand` (an activation laid out like the result) lies above the first of `bounds` and
#replaced by the second elsewhere (arrays of one float32 each): the backward pass of a ReLU
CONV_MASK = -3


def conv_tap_supported(steps_before: tp.Sequence[ConvEpilogueStep], steps_after: tp.Sequence[ConvEpilogueStep]) -> bool:
    '''The kernel stores a second result before the first step of its straight-line epilogue, or after that
    epilogue's `acc - vector` step.'''
    real = list(steps_before) + list(steps_after)
    if any(e.op == CONV_TAP for e in real) or not real or len(real) > CONV_MAX_EPI - 1:
        return False
    slots = _epilogue_template_slots(real)
    return slots != 0 and (len(steps_before) == 0 or (len(steps_before) == 1 and bool(slots & 1)))


CONV_MAX_DERIVED = 3
CONV_DERIVED_OPS = ('ADD_F', 'SUB_F', 'MUL_F', 'DIV_F', 'MAX_F', 'MIN_F', 'NEG_F', 'RSQRT_F', 'SQRT_F')


#(tag, BM, BN, threads, resident blocks per CU, relative MFMA efficiency of the tile shape)
#(efficiencies are measured: TFLOP/s of each tile on large ResNet-50 layers relative to the best)
#(128 x 128 and 128 x 64 tiles of 2 x 2 waves reached 0.92 and 0.88 of the 64 x 64 tile's rate on large layers and were
#never the estimate's choice for any shape; they are no longer built)
CONV_TILES = (('64x64', 64, 64, 256, 4, 1.00), ('32x32', 32, 32, 64, 16, 0.80))
#k steps each tile shape is built with
CONV_TILE_BK = {'64x64': (32, 64), '32x32': (32, 64)}



def choose_conv_tile(M: int, N: int, compute_units: int = 256):
    '''Smallest estimated time: tiles are dealt out over the CUs, a tile costs BM*BN / efficiency,
    and a block of one wave can drive only one of a CU's four MFMA units.'''
    if CHOICES.conv_tile is not None:
        return next(t[:4] for t in CONV_TILES if t[0] == CHOICES.conv_tile)
    best, best_time = None, None
    for tag, bm, bn, nt, occupancy, eff in CONV_TILES:
        tiles   = _cdiv(M, bm) * _cdiv(N, bn)
        #with several resident blocks per CU the tail of the last round is shared out evenly
        per_cu  = tiles / compute_units if tiles >= compute_units * occupancy else _cdiv(tiles, compute_units)
        simd    = min(1.0, (nt / 256) * min(occupancy, per_cu))
        time    = per_cu * bm * bn / (eff * simd)
        if best_time is None or time < best_time:
            best, best_time = (tag, bm, bn, nt), time
    return best


def choose_conv_split(tiles_m: int, tiles_n: int, compute_units: int = 256) -> int:
    '''How many M tiles of a layer stay 64 x 64 tiles when the rest is computed as 32 x 32 tiles (0: no split).
    tiles / CUs = 3.06 means that some CUs work on four tiles while most have three; the whole rounds keep their
    64 x 64 tiles and the remainder is spread in quarter-size units. Measured on ResNet-50 layers: +15 % at 3.06 and
    1.53 tiles per CU, +7 % at 6.1, nothing at 12.25; not used when the last round is nearly full anyway.'''
    rounds = tiles_m * tiles_n / compute_units
    whole  = int(rounds)
    if whole < 1 or rounds >= 8 or rounds - whole == 0 or rounds - whole > 0.7:
        return 0
    return (whole * compute_units) // tiles_n


def choose_conv_chunk(tiles_m: int, tiles_n: int, compute_units: int = 256) -> int:
    '''M tiles one block works through. Longer chunks hide more start-up latency (only a block's
    first tile pays for the argument fetch and the first loads); enough blocks must remain to
    keep the CUs evenly loaded.'''
    chunk = 1
    while chunk < 8 and _cdiv(tiles_m, chunk * 2) * tiles_n >= 12 * compute_units:
        chunk *= 2
    return chunk


def choose_conv_xcd_columns(M: int, N: int, K: int, tiles_m: int, tiles_n: int, lhs_size: tp.Optional[int] = None) -> int:
    '''How the tiles of a four-waves-per-tile product go to the 8 XCDs (each with an L2 of its own; workgroup b runs on XCD b % 8): 0 = consecutive
    ranges of tiles, row by row, CONV_XCD_COLUMNWISE = column by column, else 1 + log2(xn) for 8 / xn rows of xn columns of XCDs.
    Row by row an XCD with at least a row of tiles fetches the whole kernel operand, column by column the whole input: whichever fetches less.
    256 x 2048 x 2048 27.0 -> 21.3 us, 784 x 1024 x 1024 21.8 -> 20.2, 400 x 2048 x 512 11.7 -> 11.4, 196 x 2304 x 256 in four slices 8.8 -> 8.5; ResNet-50
    on six images of 160 x 160 633 -> 624 us, its training step on four of 128 x 128 2.42 -> 2.40 ms. (Column by column also where that fetches up to twice as
    much: an MLP whose wide product does, 1000 x 1000 x 700, 37.1 -> 38.7 us.) `conv_xcd_columns=None` asks for the least traffic among the rectangles
    that divide the tile grid.'''
    if CHOICES.conv_xcd_columns == 'columns':
        return CONV_XCD_COLUMNWISE
    if CHOICES.conv_xcd_columns == 'ranges':
        row, column = _cdiv(M * K if lhs_size is None else min(lhs_size, M * K), max(tiles_m, 1)), 32 * K
        each = tiles_m * tiles_n // 8
        by_rows    = row * min(tiles_m, _cdiv(each, max(tiles_n, 1))) + column * min(tiles_n, each)
        by_columns = row * min(tiles_m, each) + column * min(tiles_n, _cdiv(each, max(tiles_m, 1)))
        return CONV_XCD_COLUMNWISE if by_columns < by_rows else 0
    if (tiles_m * tiles_n) % 8:
        return 0
    if CHOICES.conv_xcd_columns is not None:
        xn = int(CHOICES.conv_xcd_columns)
        return xn.bit_length() if xn in (1, 2, 4, 8) and tiles_m % (8 // xn) == 0 and tiles_n % xn == 0 else 0
    best, best_bytes = 0, None
    for code, xn in ((1, 1), (2, 2), (3, 4), (4, 8)):
        xm = 8 // xn
        if tiles_m % xm or tiles_n % xn:
            continue
        nbytes = xn * M * K + xm * K * N
        if best_bytes is None or nbytes < best_bytes:
            best, best_bytes = code, nbytes
    return best


def choose_conv_m_blocks(tiles_m: int, tiles_n: int, compute_units: int = 256) -> int:
    '''0, or the number of blocks that share the M tiles of every N tile evenly: a grid of exactly as many blocks as
    the GPU holds at once (CHOICES.conv_blocks_per_cu per CU), each working through its tiles as one sequence of k steps, so
    that only its first tile pays for the argument fetch and the first loads. Worth it from about five tiles per
    block: with fewer, one tile more or less per block leaves CUs idle at the end (measured on ResNet-50 layers at
    batch 64: -4 to -5 % at 4.9 tiles per block, +1 to +8 % at 2.45).'''
    resident = int(CHOICES.conv_blocks_per_cu * compute_units)
    if resident < 1 or tiles_m * tiles_n < CHOICES.conv_even_split_min_tiles * resident:
        return 0
    return min(tiles_m, max(1, resident // tiles_n))


def choose_conv_bk(tag: str, g: 'ConvGeometry') -> int:
    '''The longer k step halves the barriers per MFMA. Measured on ResNet-50 layers it only pays
    for the 64x64 tile on long contractions, and only when whole k tiles stay inside one kernel
    tap (Cin % 64 == 0), which keeps the tap position in scalar registers.'''
    options = CONV_TILE_BK[tag]
    if CHOICES.conv_bk is not None and CHOICES.conv_bk in options:
        return CHOICES.conv_bk
    if tag == '64x64' and g.Cin % 64 == 0 and g.K >= 2048:
        return 64
    return 32


def _flatten_pointwise(g: ConvGeometry) -> ConvGeometry:
    '''A 1x1, stride-1, unpadded convolution over a dense feature-last array is a plain matrix
    product of the [M, Cin] pixel matrix: present it as one batch of M rows so the kernel skips
    the (batch, y, x) decode of every row.'''
    dense_in  = g.xs[3] == 1 and g.xs[1] == g.W * g.xs[2] and g.xs[0] == g.H * g.W * g.xs[2]
    dense_out = g.os == (g.Ho * g.Wo * g.N, g.Wo * g.N, g.N, 1)
    pointwise = (g.KH == g.KW == 1 and g.SH == g.SW == 1 and g.PH == g.PW == 0 and g.LH == g.LW == 1
                 and g.Ho == g.H and g.Wo == g.W)
    if not (pointwise and dense_in and dense_out) or (g.batch == 1 and g.Wo == 1):
        return g
    M = g.M
    return g._replace(batch=1, Ho=M, Wo=1, H=M, W=1, xs=(0, g.xs[2], 0, 1), os=(M * g.N, g.N, g.N, 1))


def _epilogue_template_slots(epilogue: tp.Sequence[ConvEpilogueStep]) -> int:
    '''Bit k set = step k of the kernel's straight-line epilogue (acc - vector, acc * vector,
    acc + vector, acc + full tensor, max(acc, scalar)) is present; 0 if the chain is not an
    ordered subset of those and has to go through the kernel's general step loop.'''
    template = ((EW['SUB_F'], 2, False), (EW['MUL_F'], 2, None), (EW['ADD_F'], 2, None),
                (EW['ADD_F'], 3, None), (EW['MAX_F'], 1, False))
    slots, k = 0, 0
    for e in epilogue:
        while k < len(template):
            op, kind, left = template[k]
            k += 1
            if e.op == op and e.kind == kind and (left is None or bool(e.operand_left) == left):
                slots |= 1 << (k - 1)
                break
        else:
            return 0
    return slots


def conv_straight_epilogue(epilogue: tp.Sequence[ConvEpilogueStep]) -> bool:
    return _epilogue_template_slots([e for e in epilogue if e.op != CONV_TAP]) != 0


def _magic_division(d: int) -> tp.Tuple[int, int]:
    '''(magic, shift) with n // d == (n * magic >> 32) >> shift for every 0 <= n < 2**31; magic 0 stands for d == 1.'''
    if d <= 1:
        return 0, 0
    l = (d - 1).bit_length()                  #ceil(log2(d))
    magic = -(-(1 << (31 + l)) // d)          #ceil(2**(31+l) / d) < 2**32
    return magic, l - 1


#the kernels for images of very few features: (kernel rows, values of a kernel row) -> (name, positions per tile, floats of the patch in LDS, vectors per thread)
STEM_KERNELS = {(7, 22): [('conv_gemm_stem_7x22_m128', 128, 7680, 4), ('conv_gemm_stem_7x22', 64, 6272, 6)], (3, 10): [('conv_gemm_stem_3x10_m128', 128, 7680, 4)]}


def _conv_stem_pays(g: 'ConvGeometry', tile: int, tiles: int, compute_units: int) -> bool:
    '''us there and in the general kernel, which takes its tiles across images and computes 32 columns where there are no more.'''
    filled = g.M / (tile * tiles)
    #7 x 7 x 3 to 64 features, by positions: 390 9.6, 14.2 (but test_stem_kernel_for_few_input_features promises the general one), 2601 10.1, 14.5, 72030 24.0, 32.6,
    #400000 77, 119; to 8 99225 28, 33, 400000 74, 97. Images of fewer positions than a tile: 100 of 25 9.8, 14.5, 300 of 25 15.5, 14.6, 2000 of 25 48, 26; 1000 of 64 27.8,
    #26.9, to 8 26.4, 23.2; 200 of 144 17.3, 18.3; 500 of 100 17.8, 26.9
    if g.KH == 7:
        return g.M >= 512 and (tiles <= compute_units or filled >= 0.55)
    #3 x 3 x 3. Features: 120050 positions to 8 13.9, 10.7, to 32 15.2, 12.2, to 33 15.4, 15.9, to 64 16.0, 16.6. Positions, to 64: 40000 8.8, 8.3, 69629 12.2, 12.2, 92160 12.5,
    #13.6, 175616 19.9, 21.0, 802816 55.9, 68.2; three tiles fit a CU, a few more are a second round: 94221 (754 tiles) 12.9, 13.8, 100820 (800) 15.9, 15.5, 112908 (888)
    #16.3, 15.8, 120050 (950) 16.0, 16.6. Tiles: 2000 images of 81 22.0, 19.1, 1100 of 64 16.7, 12.0, 300 of 289 14.8, 13.5, 200 of 441 15.5, 13.4, 4000 of 36 34.4, 17.5
    return g.N > 32 and g.M >= 73728 and filled >= 0.95 and not 3 < tiles / compute_units < 3.6


def _conv_stem_launch(out, lhs, rhs, g: 'ConvGeometry', epilogue, taps, compute_units, lhs_offset, rhs_offset, out_offset) -> tp.Optional[Launch]:
    '''The kernels for dense images with so few features that KW * Cin is 21 or 22 (7 x 7 x 3, seven kernel rows), or 9 or 10 (3 x 3 x 3, three), and a
    template epilogue; see the conditions listed at the kernel.'''
    #(offsets: whole images further on in both arrays - a launch over a part of the batch)
    if (CHOICES.conv_stem is False or CHOICES.conv_tile is not None or CHOICES.conv_general or rhs_offset or lhs_offset % 4 or out_offset % 4
            or (taps and (lhs_offset or out_offset))):
        return None
    M, N, K = g.M, g.N, g.K
    RL, WC = g.KW * g.Cin, g.W * g.Cin
    dense_in  = g.xs == (g.H * WC, WC, g.Cin, 1)
    dense_w   = g.ws == (g.KW * g.Cin * N, g.Cin * N, N, 1)
    dense_out = g.os == (g.Ho * g.Wo * N, g.Wo * N, N, 1)
    slots = _epilogue_template_slots(epilogue)
    left  = _cdiv(g.PW * g.Cin, 4) * 4
    right = max(0, (g.Wo - 1) * g.SW - g.PW + g.KW - g.W)          #pixels the last window reaches beyond the row
    pitch = _cdiv(left + (g.W + right) * g.Cin + 1, 4) * 4
    forms = STEM_KERNELS.get((g.KH, RL + RL % 2), [])
    if not (forms and dense_in and dense_w and dense_out and g.DH == g.DW == g.LH == g.LW == 1 and g.PH >= 0 and g.PW >= 0 and N <= 64
            and (not epilogue or (slots != 0 and not slots & 8))):
        return None
    def patch_rows(tile):                                          #the image rows that a tile's positions reach
        return (min(g.Ho, _cdiv(tile - 1, g.Wo) + 1) - 1) * g.SH + g.KH
    kernel, tile, _, _ = next((f for f in forms if (CHOICES.conv_stem != 64 or f[1] == 64) and patch_rows(f[1]) * pitch <= f[2]
                               and patch_rows(f[1]) * _cdiv(WC, 4) <= 4 * f[1] * f[3]), (None, 0, 0, 0))
    if kernel is None:
        return None
    per_image = _cdiv(g.Ho * g.Wo, tile)
    tiles     = g.batch * per_image
    if CHOICES.conv_stem is None and not _conv_stem_pays(g, tile, tiles, compute_units):
        return None
    #a second result (the value before or after the first epilogue step) goes to the last operand slot, as in conv_gemm_body
    flags  = slots << 20 | ((taps[0][0] + 1) << 12 if taps else 0)
    params = (_i32(M, N, K, g.Ho, g.Wo, g.H, g.W, g.Cin, g.KH, g.KW, g.SH, g.SW, g.PH, g.PW, pitch, left)
              + _u32(flags, (lhs.size - lhs_offset) * 4, rhs.size * 4, (out.size - out_offset) * 4, *_magic_division(per_image), *_magic_division(g.Wo))
              + _i32(tiles, per_image, patch_rows(tile)))
    derived_ptrs, derived_desc = _conv_derived(epilogue, N)
    params += derived_desc
    operand_slots = _pad([(e.operand, 0) for e in epilogue], CONV_MAX_EPI, (None, 0))
    if taps:
        assert operand_slots[-1] == (None, 0)
        operand_slots[-1] = (taps[0][1], 0)
    buffers = [(out, out_offset * 4), (lhs, lhs_offset * 4), (rhs, 0)] + operand_slots + derived_ptrs
    nbytes  = 4 * (lhs.size + rhs.size + out.size) + sum(4 * e.operand.size for e in epilogue if e.operand is not None)
    nbytes += 4 * taps[0][1].size if taps else 0
    blocks = (2 if g.KH == 7 else 4) * compute_units               #what the GPU holds at once
    return Launch(kernel, (min(tiles, blocks), 1, 1), (4 * tile, 1, 1), buffers, params, bytes_moved=nbytes, flops=2 * M * N * K)


DENSE_ROWS_MAX_N = 16
#Rows x features up to which a wave per row serves contractions that are no multiple of four: a tile for 32 rows is faster beyond (us there and by tiles: 1024 x 511 x 8 4.6, 6.3;
#5017 x 249 x 14 12.9, 5.0; 16384 x 511 x 8 36, 10; 131072 x 511 x 8 270, 57), and is as fast with multiples of four, whose sums are 2 to 3 times as far from 64 bits there
#(4096 x 256 x 10 1.5e-7, here 7.7e-8; the others came from tiles with 64-wide steps, 3.9e-7 for 64 x 511 x 8, where they are 8.8e-8)
#Of contractions that are no multiple of four: up to 32 long only this few results, because a tile takes one step for them and its epilogue any operand, which is a launch more here
#(us here and by four waves per tile; 600 x 25 x 16 4.1, 3.4, with a residual 7.2, 4.0; 4000 x 13 x 4 4.0, 3.5, 7.3, 4.1; 50 x 7 x 8 2.8, 3.1, 5.6, 3.8)
DENSE_ROWS_SHORT_RESULTS = 64
DENSE_ROWS_MAX_RESULTS = 20480


def _dense_rows_shape(lhs: Buffer, g: 'ConvGeometry') -> bool:
    '''The operands of a product suit dense_rows_n16. `g` as the caller gave it: a matrix product, not a 1 x 1
    convolution over a feature map (those keep the kernels whose epilogue takes a residual operand).'''
    if (CHOICES.conv_dense_rows is False or CHOICES.conv_tile is not None or CHOICES.conv_bk is not None or CHOICES.conv_general
            or CHOICES.conv_ksplit is not None):
        return False
    M, N, K = g.M, g.N, g.K
    flat = (g.batch == 1 and g.Wo == 1 and g.KH == g.KW == 1 and g.SH == 1 and g.PH == g.PW == 0 and g.LH == 1 and g.H == g.Ho
            and g.xs[3] == 1 and g.xs[1] >= K)
    return (flat and 1 <= N <= DENSE_ROWS_MAX_N and (K % 4 == 0 or M * N <= (DENSE_ROWS_MAX_RESULTS if K > 32 else DENSE_ROWS_SHORT_RESULTS)) and K > 0 and tuple(g.ws[2:]) == (N, 1) and tuple(g.os[1:]) == (N, N, 1)
            and lhs.size * 4 < 2**31 and M * N * 4 < 2**31)


def conv_is_dense_rows(lhs: Buffer, g: 'ConvGeometry') -> bool:
    '''This product is computed by dense_rows_n16 whatever its epilogue: a fusion pass must not hand it an epilogue that
    kernel cannot apply (another kernel would add the products in another order than in the unfused program).'''
    return g.k_splits == 1 and _dense_rows_shape(lhs, g)


def dense_rows_epilogue_supported(epilogue: tp.Sequence[ConvEpilogueStep]) -> bool:
    real  = [e for e in epilogue if e.op != CONV_SOFTMAX]
    slots = _epilogue_template_slots(real)
    return (all(e.op != CONV_TAP and e.derived is None for e in real) and (not real or (slots != 0 and not slots & 8))
            and all(e.op != CONV_SOFTMAX for e in epilogue[:-1]))


def _dense_rows_launch(out, lhs, rhs, g: 'ConvGeometry', epilogue, taps, lhs_offset, rhs_offset, out_offset,
                       softmax: bool, arg_out: tp.Optional[Buffer]) -> tp.Optional[Launch]:
    '''dense_rows_n16 where it applies: a matrix product (or 1x1 convolution over a dense array) with at most 16 output
    features and few rows, dense operands, and an epilogue of per-feature and single-value
    template steps; see the kernel.'''
    if taps or lhs_offset or rhs_offset or out_offset or g.k_splits > 1:
        return None
    M, N, K = g.M, g.N, g.K
    slots = _epilogue_template_slots(epilogue)
    if not (_dense_rows_shape(lhs, g) and dense_rows_epilogue_supported(epilogue)):
        return None
    params  = _i32(M, N, K, g.xs[1]) + _u32(slots << 20 | int(softmax) << 29, lhs.size * 4, K * N * 4, M * N * 4)
    slots_p = _pad([(e.operand, 0) for e in epilogue], CONV_MAX_EPI, (None, 0))
    if softmax:
        slots_p[-1] = (arg_out, 0)
    nbytes  = (4 * (lhs.size + rhs.size + out.size) + sum(4 * e.operand.size for e in epilogue if e.operand is not None)
               + (4 * arg_out.size if arg_out is not None else 0))
    return Launch('dense_rows_n16', (_cdiv(M, 4), 1, 1), (256, 1, 1), [(out, 0), (lhs, 0), (rhs, 0)] + slots_p, params,
                  bytes_moved=nbytes, flops=2 * M * N * K)


def _conv_derived(epilogue, N):
    '''(pointer slots, descriptor words) of the one per-feature epilogue operand that the kernel computes itself.'''
    derived_ptrs, derived_desc = [(None, 0)] * (CONV_MAX_DERIVED + 1), _u32(*[0] * (3 + 2 * CONV_MAX_DERIVED))
    for i, e in enumerate(epilogue):
        if e.derived is not None:
            d = e.derived
            assert e.kind == 2 and len(d.steps) <= CONV_MAX_DERIVED and derived_desc == _u32(*[0] * (3 + 2 * CONV_MAX_DERIVED))
            arrays = [d.first] + [st[1] for st in d.steps]
            assert all(a is None or a.size in (1, N) for a in arrays)
            derived_ptrs = _pad([(a, 0) for a in arrays], CONV_MAX_DERIVED + 1, (None, 0))
            mask = sum(1 << k for k, a in enumerate(arrays) if a is not None and a.size == N and N != 1)
            derived_desc = _u32(i, len(d.steps), mask, *_pad([st[0] for st in d.steps], CONV_MAX_DERIVED),
                                *_pad([int(st[2]) for st in d.steps], CONV_MAX_DERIVED))
    return derived_ptrs, derived_desc


def _features_in_vectors(g: ConvGeometry) -> bool:
    '''Every position's features are whole, aligned vectors of four.'''
    return g.Cin % 4 == 0 and all(s % 4 == 0 for s in g.xs[:3])


def _conv_fast_paths(lhs: Buffer, rhs: Buffer, g: ConvGeometry, lhs_offset: int = 0, rhs_offset: int = 0):
    '''(needs_masks, x_bias, a_fast, b_fast, c_contig) of a flattened geometry: which loaders and stores apply.'''
    N = g.N
    #some kernel tap of some output position falls outside the input (padding, or a window that overhangs)
    needs_masks = (g.PH > 0 or g.PW > 0 or (g.Ho - 1) * g.SH - g.PH + (g.KH - 1) * g.DH >= g.H
                   or (g.Wo - 1) * g.SW - g.PW + (g.KW - 1) * g.DW >= g.W)
    #the 16-byte A path keeps the validity of a row's taps in one 32-bit mask and addresses the
    #input from (PH, PW) positions before its start
    x_bias = (g.PH * g.xs[1] + g.PW * g.xs[2]) * 4
    #(negative padding, i.e. cropping, goes through the generic loader's coordinate checks)
    #(a vector has to start at a word only; with several taps it must not straddle two of them)
    a_fast = (g.xs[3] == 1 and (_features_in_vectors(g) or g.KH * g.KW == 1) and g.LH == 1 and g.LW == 1 and lhs_offset % 4 == 0 and g.PH >= 0 and g.PW >= 0
              and all(s >= 0 for s in g.xs[:3]) and (not needs_masks or g.KH * g.KW <= 32)
              and (lhs.size - lhs_offset) * 4 + x_bias <= 2**31)
    #16-byte loads of the kernel operand need a dense [ky, kx, in, out] array, not an output width that is a multiple of 4:
    #a buffer load of four words only has to start at a word (verified on gfx950 with integer-exact products of odd
    #widths); the words a vector reads beyond its row belong to columns >= N, which are never stored
    b_fast = (g.ws[3] == 1 and rhs_offset % 4 == 0 and not CHOICES.conv_b_general
              and g.ws[2] == N and g.ws[1] == g.Cin * N and g.ws[0] == g.KW * g.Cin * N)
    c_contig = g.os == (g.Ho * g.Wo * N, g.Wo * N, N, 1)
    return needs_masks, x_bias, a_fast, b_fast, c_contig


DENSE_COPY_MIN_K = 512
DENSE_COPY_SMALL = 14 << 20         #values


def dense_copy_applies(lhs: Buffer, g: ConvGeometry, out_size: tp.Optional[int] = None) -> bool:
    '''A kernel operand of any layout counts as a dense one, into which it may be copied first: it is no bigger than the activations, or the contraction is long. A
    step of it with element-wise loads takes 1.6 us per 32 in the general kernels and 2 per 128 where four waves share a tile, with 16-byte loads 0.65
    and 0.5; the copies of a network's kernels are one launch, at about 3 TB/s. Training steps of ResNet-50
    without and with the second clause: 8 images of 160 x 160 3.30, 2.96 ms, 4 of 96 x 96 2.28, 2.03, 5 of 224 x 224 3.39, 3.06; from 1024 on only 2.98, 2.06, 3.07,
    from 128 on 2.96, 2.03, 3.06.'''
    small = g.M >= 256 and g.K * g.N <= lhs.size + (g.M * g.N if out_size is None else out_size)
    #(operands that the kernels refuse for their size are not copied first)
    return g.N % 4 == 0 and min(g.ws) >= 0 and (small or (g.K >= DENSE_COPY_MIN_K and g.N > DENSE_ROWS_MAX_N and g.K * g.N * 4 < 2**31))


def dense_copy_pays(lhs: Buffer, g: ConvGeometry, out_size: tp.Optional[int] = None) -> bool:
    '''... and it is copied where more than one tile of rows reads it, or where it is small: the copy reads and writes it once, and takes its room in HBM. us with
    the copy, without. Transposed matrices that four waves per tile do not read as they are: 1 x 2048 x 50000 280, 223; 32 x 2048 x 50000 281, 249; 8 x 1024 x 128000
    336, 310; 64 x 768 x 30524, one row of 64 x 64 tiles, 71, 62; 64 x 512 x 30000 (61 MB) 47, 42; 64 x 2048 x 50000 318, 338; but 64 x 512 x 20000, two rows of 32 x 32,
    39, 50; 65 x 768 x 30524 92, 159; 128 x 4096 x 16384 264, 333; 256 x 2048 x 50000 612, 953. A tile of rows of a dilated input's class 25 x 512 x 8192 21, 28, x 4096 x
    1024 31, 155. Windows: 16 rows x 9216 x 1024 (38 MB) 34, 44, x 1536 (57 MB) 36, 37, x 2048 44, 43; 4 rows x 18432 x 2048 82, 79; 49 rows x 4608 x 4096 52, 76.'''
    one_tile = 32 if g.KH * g.KW != 1 else min(choose_conv_tile(g.M, g.N)[1], 64)
    return dense_copy_applies(lhs, g, out_size) and (g.M > one_tile or g.K * g.N <= DENSE_COPY_SMALL)


def _dense_kernel(g: ConvGeometry) -> bool:
    return tuple(g.ws) == (g.KW * g.Cin * g.N, g.Cin * g.N, g.N, 1)


def _kernel_operand_in_rows(g: ConvGeometry, rhs_offset: int = 0) -> bool:
    '''A transposed matrix: the four-waves-per-tile kernels read it with 16-byte loads along the contraction.'''
    return g.KH * g.KW == 1 and g.ws[2] == 1 and g.ws[3] >= 0 and rhs_offset % 4 == 0 and not CHOICES.conv_b_general


def _kernel_operand_in_vectors(lhs: Buffer, g: ConvGeometry, b_fast: bool, rhs_offset: int = 0) -> bool:
    '''For the rule of the four-waves-per-tile kernels, which read transposed matrices in vectors too: those count as dense ones where dense_copy_applies.'''
    return b_fast or (_kernel_operand_in_rows(g, rhs_offset) and dense_copy_applies(lhs, g))


def conv_reads_transposed(lhs: Buffer, rhs: Buffer, g: ConvGeometry, rhs_offset: int = 0, compute_units: int = 256) -> bool:
    '''A transposed matrix need not be copied into the dense layout: the product goes to the four-waves-per-tile kernels, as it would with the copy
    (us with the copy, without: 1000 x 100 x 300 5.9, 4.4; 1000 x 1000 x 700 21.8, 18.0; 512 x 1024 x 1024 16.6, 11.6).'''
    if not (_kernel_operand_in_rows(g, rhs_offset) and dense_copy_applies(lhs, g)):
        return False
    dense = _flatten_pointwise(g._replace(ws=(g.Cin * g.N, g.Cin * g.N, g.N, 1)))
    if _dense_rows_shape(lhs, g._replace(ws=dense.ws)) or g.K * g.N * 4 >= 2**31 or lhs.size * 4 >= 2**31:
        return False
    _, _, a_fast, _, c_contig = _conv_fast_paths(lhs, rhs, dense)
    return _four_waves_per_tile(dense, a_fast, c_contig, compute_units, True)


def _four_waves_per_tile(g: ConvGeometry, a_fast: bool, c_contig: bool, compute_units: int, b_fast: bool = True) -> bool:
    '''A product with so few 32 x 32 tiles that one wave per tile leaves most MFMA units idle: four waves per tile,
    each taking a quarter of every (128-long) k step.'''
    want = (CHOICES.conv_ksplit if CHOICES.conv_ksplit is not None else
            (CHOICES.conv_tile is None and CHOICES.conv_bk is None and _four_waves_pay(g, b_fast, compute_units)))
    return bool(want) and a_fast and c_contig and (g.Cin % 64 == 0 or g.KH * g.KW == 1) and not CHOICES.conv_general


def _four_waves_pay(g: ConvGeometry, b_fast: bool, compute_units: int) -> bool:
    '''By the rounds of one 32 x 32 tile per CU, against 64 x 64 tiles with a k step of 32 (us for M x K x N, alone):
    up to one, always (1000 x 32 x 100: 4.1 against 4.4, 196 x 64 x 512 4.1, 5.0, 196 x 224 x 512 4.8, 8.1); up to two, from a
    contraction of 64 on (784 x 32 x 512 5.1, 4.5, x 64 5.1, 5.2, x 128 5.1, 6.4, x 160 6.7, 7.1, x 256 6.7, 9.0); up to three, where
    a step of 128 that is only partly used does not cost more than it saves: 2.1 us against 0.65 for one of 32 (784 x 128 x 768 6.1,
    6.7, x 192 8.3, 8.0, x 256 8.3, 9.4, x 1024 19.6, 26.4); up to four, only long contractions (784 x 256 x 1024 9.8, 9.6, x 512
    14.6, 14.6, x 1024 23.7, 29.4). Without 16-byte loads of the kernel operand up to two
    rounds, from a contraction of 64 (200 x 16 x 1000 5.1, 4.3, x 64 5.1, 5.9, x 200 7.8, 12.2) and 128 (255 x 64 x 2048 6.7, 6.0, x 128
    8.0, 8.5). Windows from 256 on and up to two rounds, as they were measured in networks.'''
    rounds = _cdiv(_cdiv(g.M, 32) * _cdiv(g.N, 32), compute_units)
    if g.KH * g.KW != 1:
        return rounds <= 2 and g.K >= 256
    if not b_fast:
        return rounds <= 2 and g.K >= 64 * rounds
    return (rounds <= 1 or (rounds == 2 and g.K >= 64) or (rounds == 3 and 3.2 * _cdiv(g.K, 128) < _cdiv(g.K, 32))
            or (rounds == 4 and g.K >= 1024))


def conv_epilogue_is_worth_leaving_four_waves(lhs: Buffer, rhs: Buffer, g: ConvGeometry, epilogue: tp.Sequence[ConvEpilogueStep], compute_units: int = 256) -> bool:
    '''False where an epilogue would take a long product from the four-waves-per-tile kernels, which have the usual chains only: the kernel that walks
    any chain takes 0.65 us per 32 of the contraction (1.6 without 16-byte loads of the kernel operand), those 0.5 per 128, and the chain as a launch
    of its own some 4 us. (64 x 1000 x 2048, transposed kernel operand: 51.7 us, against 9.2 and 4.5.)'''
    if g.split is not None or g.k_splits > 1 or not epilogue or conv_straight_epilogue(epilogue) or _dense_rows_shape(lhs, g):
        return True
    if conv_reads_transposed(lhs, rhs, g):
        return False
    if g.K < 512:
        return True
    g = _flatten_pointwise(g)
    if g.K * g.N * 4 >= 2**31 or lhs.size * 4 >= 2**31 or g.M * g.N == 0:
        return True
    _, _, a_fast, b_fast, c_contig = _conv_fast_paths(lhs, rhs, g)
    return not (_four_waves_per_tile(g, a_fast, c_contig, compute_units, _kernel_operand_in_vectors(lhs, g, b_fast)) and (b_fast or g.Cin % 128 == 0 or g.KH * g.KW == 1))


#Up to here slices are added by a launch of their own, which also takes over chains longer than an epilogue; more tiles are shared by blocks that add them
#themselves (conv_share_count). (Shared by eight blocks, 32 tiles x 36 k steps would take 11.2 us instead of 14.4, 32 x 16 7.9 instead of 9.5; but these
#products are promised two launches: test_long_contractions_of_few_tiles_are_sliced, test_sliced_contractions.)
CONV_SLICED_MAX_TILES = 32
CONV_XCD_COLUMNWISE   = 5           #tiles go to the XCDs column by column


def conv_slicing(lhs: Buffer, rhs: Buffer, g: ConvGeometry, compute_units: int = 256) -> tp.Tuple[int, int]:
    '''(slices, shares) of a product that the four-waves-per-tile kernels compute, at most one of them above 1: into how many slices its contraction is cut that
    a launch of its own adds (conv_k_splits), and how many blocks share a tile and add theirs themselves (conv_share_count).'''
    if _dense_rows_shape(lhs, g):
        return 1, 1
    f = _flatten_pointwise(g)
    if f.K * f.N * 4 >= 2**31 or lhs.size * 4 >= 2**31 or f.M * f.N == 0:
        return 1, 1
    _, _, a_fast, b_fast, c_contig = _conv_fast_paths(lhs, rhs, f)
    #(not the 64-long step: 196 x 9 of those 7.8 us, by two blocks each 9.3)
    if not _four_waves_per_tile(f, a_fast, c_contig, compute_units, _kernel_operand_in_vectors(lhs, f, b_fast)) or (f.Cin % 128 != 0 and f.KH * f.KW != 1):
        return 1, 1
    tiles, ksteps = conv_shared_tiles(f), _cdiv(f.K, 128)
    slices = conv_k_splits(tiles, ksteps, compute_units)
    return slices, 1 if slices > 1 or g.k_splits > 1 or g.split is not None else conv_share_count(tiles, ksteps, compute_units)


def conv_k_splits(tiles: int, ksteps: int, compute_units: int = 256) -> int:
    '''Into how many slices the contraction of a product with very few tiles is cut (1: not at all). With 32 blocks on
    256 CUs, a layer whose kernel operand is megabytes long (the 3 x 3 layers of a network's last stages at batch 1)
    is bound by the rate at which those few CUs fetch it; slices spread the fetch over the chip. Every slice keeps at
    least four k steps, at most four slices (the launch that adds them is an element-wise chain with room for a
    following scale, shift and ReLU), and never more blocks than CUs.'''
    if CHOICES.conv_k_splits is not None:
        want = CHOICES.conv_k_splits
    else:
        want = 1 if tiles > CONV_SLICED_MAX_TILES else min(4, compute_units // tiles, ksteps // 4)
    if want <= 1 or ksteps < 2:
        return 1
    per = _cdiv(ksteps, min(want, ksteps))
    return _cdiv(ksteps, per)


class ConvShares(tp.NamedTuple):
    '''`count` blocks per tile, each with a slice of the contraction: they leave their sums in `partial`, and the one that finds at
    the tile's counter in `arrivals` that it is the last adds them in their order and applies the epilogue.'''
    count: int
    partial: Buffer
    arrivals: Buffer


CONV_MAX_SHARES = 8                #(of the same name in the kernel source)
CONV_MAX_SHARED_TILES = 2048


def conv_shared_tiles(g: ConvGeometry) -> int:
    return _cdiv(g.M, 32) * _cdiv(g.N, 32)


def choose_conv_shares(tiles: int, ksteps: int, compute_units: int = 256) -> int:
    '''The number of blocks per tile with the smallest estimated time. A k step of 128 takes 0.56 us alone on a CU (0.5 without masks), 1 us
    beside one other block, 1.47 beside two and 1.95 beside three, which fill a CU; those that follow start as others end. A block starts in about a
    step; leaving, counting and adding slices takes 1.6 us and 2 ns per block. Measured (tiles x k steps: one block per tile, and with the chosen number;
    the kernel operands from behind the L2s): 56 x 18 13.3, 8.5 us; 56 x 8 7.0, 6.8; 100 x 9 8.6, 8.4; 80 x 36 22.7, 12.4; 152 x 18 13.3, 11.9; 304 x 36 39.2,
    30.3 (by four blocks 34.6: a fifth on most CUs); where it stays at one, more take as long or longer: 100 x 4 5.0, 6.4; 128 x 7 6.7, 7.5; 152 x 8 7.4, 8.6;
    208 x 16 11.4, 13.5; 400 x 36 39.4, 39.1.'''
    together = (0.56, 1.0, 1.47, 1.95, 2.7, 2.95, 3.25, 3.5)
    def time(count):
        per    = _cdiv(ksteps, count)
        blocks = tiles * _cdiv(ksteps, per)
        on_cu  = _cdiv(blocks, compute_units)
        each   = together[on_cu - 1] if on_cu <= 8 else 3.5 + 0.49 * (on_cu - 8)
        return 2.9 + each * (per + 1) + (1.6 + 0.002 * blocks if count > 1 else 0.0)
    alone = time(1)
    count = min(range(1, min(ksteps, CONV_MAX_SHARES) + 1), key=time)
    return count if time(count) < 0.98 * alone else 1


def conv_share_count(tiles: int, ksteps: int, compute_units: int = 256) -> int:
    '''How many blocks share a tile (1: no sharing).'''
    pinned = CHOICES.conv_k_splits is not None or CHOICES.conv_split is not None          #(to the kernels themselves: one block per tile)
    if (CHOICES.conv_shares == 1 or tiles > CONV_MAX_SHARED_TILES
            or (CHOICES.conv_shares is None and (pinned or tiles <= CONV_SLICED_MAX_TILES))):
        return 1
    want = min(CHOICES.conv_shares, ksteps, CONV_MAX_SHARES) if CHOICES.conv_shares is not None else choose_conv_shares(tiles, ksteps, compute_units)
    return _cdiv(ksteps, _cdiv(ksteps, want))


def conv_gemm(out: Buffer, lhs: Buffer, rhs: Buffer, g: ConvGeometry, epilogue: tp.Sequence[ConvEpilogueStep] = (),
              compute_units: int = 256, lhs_offset: int = 0, rhs_offset: int = 0, out_offset: int = 0) -> Launch:
    taps = [(i, e.operand) for i, e in enumerate(epilogue) if e.op == CONV_TAP]
    if taps:
        (tap_position, tap_buffer), = taps
        epilogue = [e for e in epilogue if e.op != CONV_TAP]
        if (not conv_tap_supported(epilogue[:tap_position], epilogue[tap_position:]) or out_offset or tap_buffer.size != out.size):
            raise ValueError('a second result at this point of the epilogue is not supported')
    softmax, arg_out = False, None
    if epilogue and epilogue[-1].op == CONV_SOFTMAX:
        softmax, arg_out = True, epilogue[-1].operand
        epilogue = list(epilogue[:-1])
        if len(epilogue) > CONV_MAX_EPI - 1 or (arg_out is not None and arg_out.size != g.M):
            raise ValueError('softmax epilogue: too many steps, or labels of another size')
    if any(e.op == CONV_SOFTMAX for e in epilogue):
        raise ValueError('softmax can only be the last step of an epilogue')
    if len(epilogue) > CONV_MAX_EPI:
        raise ValueError('too many epilogue steps')
    g_given, g = g, _flatten_pointwise(g)
    M, N, K = g.M, g.N, g.K
    for name, extent in (('lhs', lhs.size), ('rhs', rhs.size), ('out', out.size)):
        if extent * 4 >= 2**31:
            raise NotImplementedError(f'conv/dot {name} operand of {extent * 4} bytes exceeds the 2 GiB the kernel addresses')
    rows = _dense_rows_launch(out, lhs, rhs, g_given, epilogue, taps, lhs_offset, rhs_offset, out_offset, softmax, arg_out)
    if rows is not None:
        return rows
    if softmax:
        raise ValueError('softmax epilogue: only in the kernel for at most 16 output features')
    stem = _conv_stem_launch(out, lhs, rhs, g, epilogue, taps, compute_units, lhs_offset, rhs_offset, out_offset)
    if stem is not None:
        return stem
    tag, bm, bn, nt = choose_conv_tile(M, N, compute_units)
    bk = choose_conv_bk(tag, g)
    needs_masks, x_bias, a_fast, b_fast, c_contig = _conv_fast_paths(lhs, rhs, g, lhs_offset, rhs_offset)
    slots = _epilogue_template_slots(epilogue)
    #One step of a contraction that is no multiple of four, and a large full tensor behind it: all of it is time in memory, and the kernels that load word by word overlap
    #that better than those that fetch the tensor a tile ahead (us by vectors and words: 255921 x 13 x 104 60.7, 49.4; 230625 x 6 x 104 52.9, 44.0; 221664 x 13 x 24 22.0, 17.3;
    #24088 x 5 x 256 14.3, 13.4; but 40426 x 6 x 104 11.4, 11.9; 73931 x 5 x 48 10.8, 11.8; 179393 x 33 x 64 28.7, 31.2)
    if K % 4 != 0 and K <= 32 and slots & 8 and M * N >= 5 << 20:
        a_fast = False
    #the lean kernel variant covers the common case only (see the kernel source)
    lean = (a_fast and b_fast and c_contig and (g.Cin % bk == 0 or g.KH * g.KW == 1)
            and (not epilogue or slots != 0) and not CHOICES.conv_general)
    #the output row number is the input row number (a matrix product, or a one-column image walked without stride,
    #padding or taps outside the input): the kernel then skips the row decode and the validity masks
    flat_rows = g.batch == 1 and g.Wo == 1 and g.SH == 1 and g.PH == 0 and g.PW == 0 and not needs_masks
    #a product with so few 32 x 32 tiles that one wave per tile leaves most MFMA units idle: four waves per
    #tile, each taking a quarter of every (128-long) k step
    ksplit = _four_waves_per_tile(g, a_fast, c_contig, compute_units, _kernel_operand_in_vectors(lhs, g, b_fast, rhs_offset)) and (not epilogue or slots != 0)
    #(windows over 64 input features take a 64-long k step, with 16-byte loads of the kernel operand only)
    short_step = ksplit and g.Cin % 128 != 0 and g.KH * g.KW != 1
    if short_step and not b_fast:
        ksplit = False
    #results whose rows lie apart, without an epilogue and with dense kernel operands: the same by strides
    strided = (not ksplit and not c_contig and b_fast and not epilogue and not taps and g.k_splits == 1 and min(g.os) >= 0
               and (g.Cin % 32 == 0 or g.KH * g.KW == 1) and _four_waves_per_tile(g, a_fast, True, compute_units, True))
    ksplit = ksplit or strided
    if strided:
        short_step = False
    if ksplit:
        tag, bm, bn, nt, bk, lean = '32x32', 32, 32, 256, 64 if short_step else 128, True
    tiles_m, tiles_n = _cdiv(M, bm), _cdiv(N, bn)
    k_split_steps = 0
    if g.k_splits > 1:
        k_split_steps = _cdiv(_cdiv(K, 128), g.k_splits)
        if (not ksplit or short_step or epilogue or taps or out_offset or out.size != g.k_splits * M * N
                or _cdiv(_cdiv(K, 128), k_split_steps) != g.k_splits):
            raise ValueError('a sliced contraction needs the four-waves-per-tile kernel, no epilogue and one [M, N] matrix per non-empty slice')
    elif g.shares is not None and ksplit and not short_step and not strided:
        k_split_steps = _cdiv(_cdiv(K, bk), g.shares.count)
        if (out_offset or _cdiv(_cdiv(K, bk), k_split_steps) != g.shares.count or tiles_m * tiles_n > g.shares.arrivals.size
                or g.shares.partial.size < tiles_m * tiles_n * g.shares.count * 1024):
            raise ValueError('shared tiles need a whole result, a non-empty slice for every block, and scratch for all of them')
    chunk = (CHOICES.conv_chunk or choose_conv_chunk(tiles_m, tiles_n, compute_units)) if lean and not ksplit else 1
    m_blocks = 0
    if lean and not ksplit and CHOICES.conv_chunk is None:
        m_blocks = choose_conv_m_blocks(tiles_m, tiles_n, compute_units)
        if m_blocks:
            chunk = 2                          #(a value other than 1 keeps the mixed tiling out; the kernel ignores it)
    #64 x 64 tiles that do not divide evenly among the CUs: as many M tiles as fill every CU equally stay 64 x 64, the
    #rows behind them are computed as 32 x 32 tiles with four waves per tile (a quarter of the work each)
    split_tiles_m = 0
    mixable = (lean and not ksplit and tag == '64x64' and chunk == 1 and b_fast and (g.Cin % 64 == 0 or g.KH * g.KW == 1) and K >= 256)
    if mixable and CHOICES.conv_mix is not None and CHOICES.conv_mix is not False:
        split_tiles_m = int(CHOICES.conv_mix)                      #tests: whatever the other pinned choices are
    elif mixable and CHOICES.conv_mix is None and CHOICES.conv_tile is None and CHOICES.conv_bk is None and CHOICES.conv_chunk is None:
        split_tiles_m = choose_conv_split(tiles_m, tiles_n, compute_units)
    if split_tiles_m >= tiles_m:
        split_tiles_m = 0
    kinds = [e.kind for e in epilogue]
    x_bytes = (lhs.size - lhs_offset) * 4
    w_bytes = K * N * 4 if b_fast else (rhs.size - rhs_offset) * 4
    first_full = kinds.index(3) + 1 if 3 in kinds else 0
    flags = (int(c_contig) | int(flat_rows) << 1 | int(needs_masks) << 2 | len(epilogue) << 8 | first_full << 16
             | slots << 20 | chunk << 25 | ((tap_position + 1) << 12 if taps else 0))
    if ksplit:
        flags |= choose_conv_xcd_columns(M, N, K, tiles_m, tiles_n, lhs.size - lhs_offset) << 29
    descs = [0, 0]
    for i, e in enumerate(epilogue):
        assert e.op < 128 and 1 <= e.kind <= 3
        descs[i // 3] |= ((e.op * 2 + int(e.operand_left)) | e.kind << 8) << (10 * (i % 3))
    slices = g.shares.count if k_split_steps and g.k_splits == 1 else g.k_splits
    #the kernels whose four waves share a tile divide by multiplying; they need no strides of the result and no dilation of the input
    dilation, out_strides, per_block = _i32(g.LH, g.LW), _i32(*g.os), _i32(tiles_m // m_blocks if m_blocks else 0)
    if ksplit or split_tiles_m:
        rows, columns = (tiles_m, tiles_n) if ksplit else (_cdiv(M - split_tiles_m * 64, 32), _cdiv(N, 32))
        dilation, per_block = _u32(*_magic_division(g.Cin)), _i32(slices)
        out_strides = _u32(*_magic_division(rows if flags >> 29 == CONV_XCD_COLUMNWISE else columns), *_magic_division(rows * columns))
    params = (_i32(M, N, K, g.Ho, g.Wo, g.H, g.W, g.Cin, g.KH, g.KW, g.SH, g.SW, g.PH, g.PW, g.DH, g.DW,
                   *g.xs[:3], tiles_m, tiles_n)
              #(rows beyond M are dropped by the descriptor's size: with slices, that of one slice's matrix)
              + _u32(flags, *descs, x_bytes, w_bytes, M * N * 4 if k_split_steps else (out.size - out_offset) * 4,
                     *_magic_division(g.Ho * g.Wo), *_magic_division(g.Wo))
              + dilation + _i32(g.xs[3], *(g.os if strided else g.ws)) + out_strides + _i32(split_tiles_m, k_split_steps, m_blocks) + per_block + _i32(tiles_m % m_blocks if m_blocks else 0))
    derived_ptrs, derived_desc = _conv_derived(epilogue, N)
    params += derived_desc
    buffers = [(out, out_offset * 4), (lhs, lhs_offset * 4), (rhs, rhs_offset * 4)]
    shared  = k_split_steps > 0 and g.k_splits == 1
    if shared:
        buffers += [(g.shares.partial, 0), (g.shares.arrivals, 0)]
    operand_slots = _pad([(e.operand, 0) for e in epilogue], CONV_MAX_EPI, (None, 0))
    if taps:
        assert operand_slots[-1] == (None, 0)
        operand_slots[-1] = (tap_buffer, 0)
    buffers += operand_slots + derived_ptrs
    kernel  = f'conv_gemm_{tag}x{bk}_' + (('ks4_strided' if strided else 'ks4' if b_fast else 'ks4t' if _kernel_operand_in_rows(g, rhs_offset) else 'ks4g') + ('_shared' if shared else '') if ksplit else 'lean' if lean else ('f' if a_fast else 'g') + ('f' if b_fast else 'g'))
    nbytes  = 4 * (lhs.size + rhs.size + out.size) + sum(4 * e.operand.size for e in epilogue if e.operand is not None)
    nbytes += 4 * tap_buffer.size if taps else 0
    blocks = (m_blocks or _cdiv(tiles_m, chunk)) * tiles_n * slices
    if split_tiles_m:
        kernel = f'conv_gemm_{tag}x{bk}_mix'
        blocks = split_tiles_m * tiles_n + _cdiv(M - split_tiles_m * 64, 32) * _cdiv(N, 32)
    return Launch(kernel, (blocks, 1, 1), (nt, 1, 1), buffers, params, bytes_moved=nbytes, flops=2 * M * N * K,
                  written=(0, 3, 4) if shared else (0,), scratch=(3, 4) if shared else ())


# ------------------------------------------------- products on the bf16 matrix cores (csrc/kernels/conv_split.h)

#tile -> (BM, BN, microseconds of a CU per k tile of 32: with several blocks on it, with one)
CONV_SPLIT_TILES = {'128x128': (128, 128, 1.15, 1.15), '128x64': (128, 64, 0.65, 0.95)}
#tile -> microseconds of a CU per k tile of 32 for the kernels that hold a patch of the input in LDS, and what a block's start and end cost, and those
#of a slice, in k tiles. (Products alone, 128x64 and 128x128: 64 x 28 x 28 x 128 x 128 74.7 in 832 blocks and 75.9, 64 x 14 x 14 x 256 x 256 78.7, 75.2, 64 x 7 x 7
#x 512 x 512 80.1, 78.1 in 200 blocks, 16 x 7 x 7 x 512 x 512 73.9 in 56 blocks, 41.8 in 112, 29.2 in 224; 119, 66, 41.)
CONV_PATCH_STEP, CONV_PATCH_START, CONV_PATCH_SLICE = {'128x128': 0.88, '128x64': 0.5, 'fine': 0.65}, 8, 16
#Products below these stay with the fp32 kernels. Rows: packing the kernel operand costs what about 250 rows' products cost,
#and one launch. Contraction: with two k tiles of 32 a block is all start-up and stores (12544 x 64 x 256 with residual 29
#us here, 25 there; 200704 x 64 x 256 115, 113, and 0.8 times that where a block holds the kernel operand, _conv_short_pays; 50176 x 128 x 512: 59 against 61). Operations: start and end of two launches. A
#product alone is slower up to 2 GFLOP (8188 x 880 x 98, 1.4: 28.9 against 23.9; 20000 x 512 x 64, 1.3: 23.4, 21.6; 8192 x 512 x 256, 2.1: 23.0,
#23.4), by the packing launch; in a network, where several layers' weights are packed by one launch, it is faster from 1 on, more so where
#the backward pass of a ReLU is its epilogue (ResNet-50 with the line at 1, at 1.5 and at 2: batch 16 1566, 1583, 1623 us, batch 8 at 200 x 200 1092, 1119,
#1120; its training step at batch 16 5603, 5577, 5976, at batch 24 on 160 x 160 5099, 5407, 5408).
CONV_SPLIT_MIN_M, CONV_SPLIT_MIN_K, CONV_SPLIT_MIN_FLOPS = 2049, 128, 1e9
CONV_SPLIT_ROUND = 256             #tiles of a whole round, one per CU; only those behind the last whole round are shared, fewer than this many
CONV_SPLIT_MASKED = 1 << 25        #ConvParams.flags: the epilogue has a mask (conv_masked_epilogue)
CONV_SPLIT_PACK_BYTES = 12288      #packed kernel operand: bytes per 32 columns and pair of k tiles of 32


class ConvSplit(tp.NamedTuple):
    '''How a product is shared out: the first `whole` tiles of the grid by one block each, the contraction of every tile
    behind them by `slices` blocks. Those leave their sums in `partial`, and the one that finds at the tile's counter in
    `arrivals` that it is the last adds them.'''
    tile: str
    whole: int
    slices: int
    partial: tp.Optional[Buffer] = None
    arrivals: tp.Optional[Buffer] = None
    patch: bool = False               #by the kernels that hold a patch of the input in LDS (conv_patch_applies)
    ragged: bool = False              #... of any number of features, with two sums (conv_ragged_applies)
    fine: bool = False                #... by the one with two sums (_conv_patch_pays)
    short: bool = False               #by the kernels that hold the kernel operand in LDS (conv_short_applies)


def conv_split_tiles(split: ConvSplit, g: ConvGeometry) -> tp.Tuple[int, int]:
    bm, bn = CONV_SPLIT_TILES[split.tile][:2]
    return _cdiv(g.M, bm), _cdiv(g.N, bn)


def conv_split_partial_words(split: ConvSplit, g: ConvGeometry) -> int:
    bm, bn = CONV_SPLIT_TILES[split.tile][:2]
    tiles_m, tiles_n = conv_split_tiles(split, g)
    return (tiles_m * tiles_n - split.whole) * split.slices * bm * bn * (2 if split.fine else 1)


def conv_split_packed_words(g: ConvGeometry) -> int:
    if g.split is not None and g.split.patch:
        return _cdiv(g.N, 32) * (conv_patch_k(g) // 32) * (CONV_SPLIT_PACK_BYTES // 8)
    return _cdiv(g.N, 32) * _cdiv(g.K, 64) * (CONV_SPLIT_PACK_BYTES // 4)


def conv_patch_k(g: ConvGeometry) -> int:
    '''The contraction as the kernels that hold a patch walk it: features in pairs of sixteens.'''
    return g.KH * g.KW * _cdiv(g.Cin, 32) * 32


def conv_ragged_applies(g: ConvGeometry) -> bool:
    '''3 x 3 windows at a stride of 1 over dense images with a border of one: the positions of a tile and their neighbours are
    consecutive in memory. A patch has room for 256 positions (128 + 2 W + 2).'''
    return ((g.KH, g.KW, g.SH, g.SW, g.PH, g.PW, g.DH, g.DW, g.LH, g.LW) == (3, 3) + (1,) * 8
            and g.Ho == g.H and g.Wo == g.W and g.W <= 63 and g.Cin >= 4 and g.xs[2] >= g.Cin and g.xs[3] == 1
            and g.xs[1] == g.W * g.xs[2] and g.xs[0] == g.H * g.xs[1])


def conv_patch_applies(g: ConvGeometry) -> bool:
    return conv_ragged_applies(g) and g.Cin % 32 == 0


def conv_short_applies(g: ConvGeometry, c_contig: bool) -> bool:
    '''Dense rows of at most 64 features (a flattened geometry), the result's rows dense too.'''
    #(the kernel has no stride along the contraction: an operand that is contracted over its rows is not for it; nor does it clear what the last vector
    #of a row that is no whole number of them holds of the next row, which zeros on the other side would not keep out where it is not finite)
    return (c_contig and 0 < g.K <= 64 and g.xs[3] == 1 and g.xs[1] >= g.K and _features_in_vectors(g) and (g.KH, g.KW, g.SH, g.SW, g.PH, g.PW, g.LH, g.LW) == (1,) * 4 + (0,) * 2 + (1,) * 2
            and g.batch == 1 and g.Wo == 1 and g.Ho == g.H)


def _conv_short_pays(g: ConvGeometry) -> bool:
    '''Where those kernels are faster than any other.'''
    #(times of replays of a product with a residual behind its ReLU in microseconds, packing included, fp32 and here.) Columns: half lines of a width
    #that is no multiple of 32 are requested twice (43000 x 64 x 300 35, 41; 100000 x 48 x 300 80, 76), and below 96 there is little to walk (200704 x 64 x 64 32, 34). Features: 200704 x 36 x 256 101, 79, but without an epilogue 200704
    #x 32 x 256 50, 57. Results: 10 M 40000 x 64 x 256 26, 29; 12.8 M 100352 x 64 x 128 31, 32; 17 M 65536 x 64 x 256 41, 34, 131072 x 64 x 128 40, 34, 8200 x
    #64 x 2048 40, 36 (without an epilogue 30, 30); 19 M 200704 x 64 x 96 66, 42. With the backward pass of a ReLU half as long from 12 M on
    return g.N % 32 == 0 and g.N >= 96 and g.K > 32 and g.M * g.N >= 1 << 24


def _conv_ragged_pays(g: ConvGeometry, dense: bool, copied: bool) -> bool:
    '''3 x 3 windows over a number of features that is no multiple of 32, for which the fp32 kernels look every vector's tap up (or, without whole
    vectors, every word's): where the kernel that holds a patch, whose errors are no larger, is faster, its packing launch included (us there and here).
    `dense`: the kernel operand is laid out as those load it in vectors; `copied`: it would be copied into that layout for them.'''
    one_round = 200 <= _cdiv(g.M, 64) * _cdiv(g.N, 64) <= 256           #their 64 x 64 tiles keep every CU busy once
    flops     = 2 * g.M * g.N * g.K
    #loads of words, images x size, features: 1 x 8, 22 15.8, 13.1; 60 x 40, 22 37.7, 27.8; 30 x 14, 41 25.3, 18.2; 11 x 31, 397 589, 209; 3 x 22, 417 219, 55; but 4 x 14, 17
    #12.5, 13.5; 60 x 40, 9 18.5, 26.7; in one round 4704 x 33 to 152 22.4, 23.5
    if g.Cin % 4 != 0:
        return g.Cin >= 20 and not (dense and one_round and 33 <= g.Cin <= 36)
    #Of vectors, another layout of the kernel operand (that of an input gradient, often with the backward pass of a ReLU behind it, which is part of the launch here): by words 336 x
    #76 to 288 34, 19; 29602 x 52 to 78 69, 34; 11520 x 80 to 306 101, 51; but 128000 x 4 to 286 153, 158; copied 21660 x 40 to 144 48, 37; but 231125 x 80 to 8 121, 137
    if not dense:
        return ((g.Cin >= 100 and (g.N >= 24 or g.M <= 8192)) or (g.Cin >= 60 and g.M <= 1024)
                or (g.Cin >= 12 and flops >= 1.5e9 and not (copied and g.N <= 32 and g.Cin < 144)))
    #the dense one; a long contraction (1 x 8, 104 27.7, 18.3; 64 x 7, 200 50, 39; 16 x 14, 136 35, 29), but not where those compute no column too many (60 x 28, 100 to 17 43.5,
    #47.6; 46550 x 100 to 32 43.5, 48; 18252 x 104 to 24 30, 33; 15984 x 152 to 24 39, 34), nor in one round where a sixth of the features is padding (3240 x 104 to 264 33, 36; 2704
    #x 132 to 296 35, 38; 6727 x 120 to 120 31.6, 29.3), ...
    times = _cdiv(g.Cin, 32) * 32 / g.Cin
    if g.Cin >= 100:
        if g.Cin < 144 and ((one_round and times >= 1.2) or (g.N <= 32 and g.M > 8192)):
            return False
        if g.N >= 24 or g.M <= 8192:
            return True
    #... few positions (4 x 14, 60 18.1, 16.9; 4 x 14, 80 22.6, 18.3; but 560 x 68 to 272 20.8, 21.8, 30 x 14, 72 21.7, 25.3), or many operations (60 x 40, 60
    #71.9, 53.2; 2888 x 92 to 344 33, 29; 112896 x 240 to 8 171, 165; but 10 x 40, 60 20.0, 25.0), more of them where much is padding (54692 x 8 to 288 48, 76; 49572 x 36 to 88 45,
    #51; 9438 x 40 to 224 30, 32; 8100 x 68 to 360 43, 49; 20800 x 68 to 68 34, 38; but 24986 x 44 to 216 58, 54, 25596 x 68 to 68 44.7, 41.7, 68400 x 68 to 112 126, 99), and not for
    #up to 32 columns, which those do not pad (312852 x 72 to 4 137, 172; 197843 x 52 to 24 77, 96; 75625 x 80 to 32 49, 55); to 64, which they do, from fewer features on (96000 x 36 to 36
    #47.8, 43.5; 57154 x 40 to 40 35, 33.5; but 66248 x 36 to 36 37, 40), or from more operations on (62424 x 40 to 328 176, 161)
    return ((g.Cin >= 60 and times < 1.35 and g.M <= 1024) or (g.Cin >= 144 and flops >= 1.5e9)
            or (g.Cin >= 44 and g.N > 32 and flops >= (4e9 if times >= 1.35 and g.M < 24576 else 1.5e9))
            or (g.Cin >= 36 and g.N > 32 and flops >= (1.6e9 if g.N <= 64 else 8e9)))


def _conv_patch_pays(g: ConvGeometry, c_contig: bool) -> bool:
    '''Products that stay with the fp32 kernels otherwise: where the kernel that holds a patch and keeps two sums, whose errors are no larger than
    theirs however few of a sum's terms are not zero, is faster than they are, packing included (images x H x W x features x columns: there, here).'''
    flops = 2 * g.M * g.N * g.K
    #16 x 7 x 7 x 512 x 512 (3.7 GFLOP) 48, 45; 33 x 7 x 7 x 512 x 512 101, 67; 64 x 56 x 56 x 64 x 32 114, 86; but 18 x 6 x 6 x 512 x 512 (3.1) 48, 49; 8 x 7 x 7 x 512
    #x 512 (1.9) 31, 38; of 32 features 32 x 56 x 56 x 32 x 32 26, 32
    if flops >= 3.5e9:
        return g.K >= 576
    #four waves that share a contraction are as fast or faster: 4 x 28 x 28 x 128 x 128 16, 23; 8 x 14 x 14 x 256 x 256 27, 32; 10 x 10 x 10 x 320 x 320 33, 35
    if _four_waves_per_tile(g, True, c_contig, CONV_SPLIT_ROUND):
        return False
    #one wave walks the whole contraction there: 1 x 7 x 7 x 480 x 480 93, 32; 3 x 13 x 13 x 224 x 224 45, 25; 1 x 10 x 10 x 160 x 40 33, 18; 1519 rows x 160 x 308 35, 32;
    #of 96 features 1 x 7 x 7 x 96 x 96 21, 17; 2673 rows x 96 x 97 (84 tiles) 22, 20, 3600 x 96 x 96 (114) 22, 22, 16200 x 96 x 32 22, 26; of 64 4 x 56 x 56 x 64 x 64 16, 21
    return g.K >= 1440 or (g.K >= 864 and _cdiv(g.M, 64) * _cdiv(g.N, 64) <= 96)


def _conv_split_pays(g: ConvGeometry, c_contig: bool) -> bool:
    '''Where the kernels on the bf16 matrix cores are faster than the fp32 kernels that would compute the product otherwise.'''
    M, N, K = g.M, g.N, g.K
    if M < CONV_SPLIT_MIN_M or K < CONV_SPLIT_MIN_K or 2 * M * N * K < CONV_SPLIT_MIN_FLOPS:
        return False
    #(times in microseconds, here and there)
    if N <= 32:
        #half of a tile is columns that do not exist: 65536 x 1024 x 32 58, 48; 16384 x 4096 x 32 70, 49; 50176 x 4096 x 32 202, 185. Except where
        #the fp32 tiles are more than four waves share and fewer than the SIMDs: 20000 x 2048 x 32 42, 55; 30000 x 4096 x 32 122, 161
        return K >= 2048 and 2 * CONV_SPLIT_ROUND < _cdiv(M, 32) <= 4 * CONV_SPLIT_ROUND
    #short and narrow: bound by HBM on both sides, start and end of a block count (65536 x 128 x 64 18, 15; 157776 x 136 x 63 39, 36; 200704 x 128 x 64
    #40, 41, with a residual behind its ReLU 51, 45; 65536 x 192 x 64 22, 20; 200704 x 192 x 64 47, 49)
    if N <= 64 and K < 192:
        return False
    #few tiles: the fp32 kernel whose four waves share a tile is ahead until the contraction is long (K = 2048, 4096 and 8192: 4096 x 64 22, 16;
    #31, 27; 46, 48. 4096 x 128 31, 24; 42, 43; 64, 80. 3136 x 128 33, 24; 44, 41; 59, 76)
    return K >= 4096 or _cdiv(M, 32) * _cdiv(N, 32) > 2 * CONV_SPLIT_ROUND or not _four_waves_per_tile(g, True, c_contig, CONV_SPLIT_ROUND)


def conv_split_plan(lhs: Buffer, g: ConvGeometry) -> tp.Optional[ConvSplit]:
    '''The plan with the smallest estimated time, or None where these kernels do not apply or another one is faster.'''
    if (CHOICES.conv_split is False or g.k_splits > 1 or _dense_rows_shape(lhs, g) or CHOICES.conv_general or CHOICES.conv_b_general
            or any(v is not None for v in (CHOICES.conv_tile, CHOICES.conv_bk, CHOICES.conv_chunk, CHOICES.conv_ksplit, CHOICES.conv_k_splits, CHOICES.conv_mix))
            or CHOICES.conv_stem not in (None, True)):
        return None
    g = _flatten_pointwise(g)
    M, N, K = g.M, g.N, g.K
    _, _, a_fast, _, c_contig = _conv_fast_paths(lhs, lhs, g, 0)
    #(features that k tiles of 32 divide, or a single tap; one of the kernels that hold a patch takes any number)
    tiled = a_fast and _features_in_vectors(g) and (g.Cin % 32 == 0 or g.KH * g.KW == 1)
    if M * N == 0 or _cdiv(N, 32) * g.KH * g.KW * _cdiv(g.Cin, 32) * (CONV_SPLIT_PACK_BYTES // 2) >= 2**31:
        return None
    #(pinned to other kernels of this family, a product is theirs)
    wanted = CHOICES.conv_split is None and CHOICES.conv_split_slices is None if CHOICES.conv_patch is None else CHOICES.conv_patch
    patch  = bool(wanted) and conv_patch_applies(g)
    wanted = CHOICES.conv_split is None and CHOICES.conv_split_slices is None if CHOICES.conv_short is None else CHOICES.conv_short
    if wanted and conv_short_applies(g, c_contig) and (CHOICES.conv_short or _conv_short_pays(g)):
        return ConvSplit('128x64', _cdiv(M, 128) * _cdiv(N, 64), 1, short=True)
    ragged = (conv_ragged_applies(g) and not patch and CHOICES.conv_split is None and CHOICES.conv_split_slices is None
              and (CHOICES.conv_ragged if CHOICES.conv_ragged is not None else _conv_ragged_pays(g, _dense_kernel(g), dense_copy_pays(lhs, g))))
    if not tiled and not ragged:
        return None
    if ragged:
        patch = True
    pays  = tiled and _conv_split_pays(g, c_contig)
    fine  = ragged or patch and (CHOICES.conv_patch == 'fine' or (CHOICES.conv_patch is None and not pays))
    if not (ragged or CHOICES.conv_split or CHOICES.conv_split_slices or (patch and CHOICES.conv_patch)) and not (_conv_patch_pays(g, c_contig) if fine else pays):
        return None
    #The whole tiles are dealt out in rounds of one per CU; the contraction of those of the last, incomplete round (or of all,
    #if there are fewer tiles than CUs) may be cut into slices, of two k tiles at least. A block's start and end cost about
    #three k tiles, a slice's partial sums five more (a patch has to be complete before the first product: eight).
    ktiles, best = conv_patch_k(g) // 32 if patch else 2 * _cdiv(K, 64), None
    for tile, (bm, bn, shared_step, lone_step) in CONV_SPLIT_TILES.items():
        if CHOICES.conv_split not in (None, True, tile) or (fine and tile != '128x64'):
            continue
        tiles = _cdiv(M, bm) * _cdiv(N, bn)
        for slices in range(1, 17):
            whole = tiles if slices == 1 else tiles // CONV_SPLIT_ROUND * CONV_SPLIT_ROUND
            if slices > 1 and (ktiles < (9 if patch else 2) * slices or whole == tiles) or CHOICES.conv_split_slices not in (None, slices):
                continue
            blocks = whole + (tiles - whole) * slices
            rounds = whole / CONV_SPLIT_ROUND if slices > 1 else _cdiv(tiles, CONV_SPLIT_ROUND)
            step   = CONV_PATCH_STEP['fine' if fine else tile] if patch else shared_step if blocks > CONV_SPLIT_ROUND else lone_step
            start, slice_start = (CONV_PATCH_START, CONV_PATCH_SLICE) if patch else (3, 8)
            time   = step * (rounds * (ktiles + start) + _cdiv((tiles - whole) * slices, CONV_SPLIT_ROUND) * (ktiles / slices + slice_start))
            if best is None or time < best[0]:
                best = (time, ConvSplit(tile, whole, slices, patch=patch, ragged=ragged, fine=fine))
    return best[1] if best else None


def conv_split_pack(packed: Buffer, source: EwOperand, g: ConvGeometry) -> Launch:
    '''The kernel operand of a product, element (ky, kx, c, n) at source.offset + (ky, kx, c, n) . source.strides, taken
    apart into three bf16 parts and laid out for the matrix cores.'''
    assert packed.size == conv_split_packed_words(g)
    patch  = g.split is not None and g.split.patch
    params = _i32(g.N, -conv_patch_k(g) if patch else g.K, g.Cin, g.KW, *source.strides)
    blocks = _cdiv(_cdiv(g.N, 32) * (conv_patch_k(g) // 16), 4) if patch else _cdiv(g.N, 32) * _cdiv(g.K, 64)
    return Launch('conv_split_pack', (blocks, 1, 1), (BLOCK, 1, 1), [(packed, 0), (source.buffer, source.offset * 4)], params,
                  bytes_moved=4 * (packed.size + g.K * g.N))


def conv_split_launch(out: Buffer, lhs: Buffer, packed: Buffer, g: ConvGeometry, epilogue: tp.Sequence[ConvEpilogueStep] = (),
                      lhs_offset: int = 0, out_offset: int = 0) -> Launch:
    split, g = g.split, _flatten_pointwise(g)
    M, N, K  = g.M, g.N, g.K
    needs_masks, _, _, _, c_contig = _conv_fast_paths(lhs, lhs, g, lhs_offset)
    flat_rows = g.batch == 1 and g.Wo == 1 and g.SH == 1 and g.PH == 0 and g.PW == 0 and not needs_masks
    flags     = int(c_contig) | int(flat_rows) << 1 | int(needs_masks) << 2
    taps = [(i, e.operand) for i, e in enumerate(epilogue) if e.op == CONV_TAP]
    masked = any(e.op == CONV_MASK for e in epilogue)
    if masked:
        operands = conv_masked_epilogue(epilogue)
        if operands is None or out_offset or any(e.operand.size != out.size for e in epilogue if e.kind == 3):
            raise ValueError('an epilogue with a mask is: + full tensor, mask, second result, * vector')
        flags   |= CONV_SPLIT_MASKED | len(taps) << 12
        epilogue = [e or ConvEpilogueStep(EW['NOP'], 0, None) for e in operands]
    elif taps:
        (tap_position, tap_buffer), = taps
        epilogue = [e for e in epilogue if e.op != CONV_TAP]
        if not conv_tap_supported(epilogue[:tap_position], epilogue[tap_position:]) or out_offset or tap_buffer.size != out.size:
            raise ValueError('a second result at this point of the epilogue is not supported')
        flags |= (tap_position + 1) << 12
    slots = (8 if epilogue[0].operand is not None else 0) | (2 if epilogue[2].operand is not None else 0) if masked else _epilogue_template_slots(epilogue)
    steps = bool(epilogue) and not slots and not masked           #any other chain: the kernel that walks through its steps
    if steps and taps:
        raise ValueError('a second result at this point of the epilogue is not supported')
    for name, extent in (('lhs', lhs.size), ('packed rhs', packed.size), ('out', out.size)):
        if extent * 4 >= 2**31:
            raise NotImplementedError(f'conv/dot {name} operand of {extent * 4} bytes exceeds the 2 GiB the kernel addresses')
    kinds  = [e.kind for e in epilogue]
    flags |= len(epilogue) << 8 | ((int(bool(slots & 8)) if masked else kinds.index(3) + 1) if 3 in kinds else 0) << 16 | slots << 20
    descs  = [0, 0]
    for i, e in enumerate(epilogue):
        descs[i // 3] |= ((0 if masked else e.op * 2 + int(e.operand_left)) | e.kind << 8) << (10 * (i % 3))
    (tiles_m, tiles_n), kpairs = conv_split_tiles(split, g), _cdiv(g.Cin, 32) if split.patch else _cdiv(K, 64)
    assert not split.patch or (conv_ragged_applies if split.ragged else conv_patch_applies)(g)
    shared = tiles_m * tiles_n - split.whole
    blocks, threads, kernel = split.whole + shared * split.slices, 256, f'conv_gemm_split_{split.tile}' + ('_ragged' if split.ragged else ('_patch' if split.patch else '') + ('_fine' if split.fine else ''))
    if split.short:
        assert conv_short_applies(g, c_contig) and flat_rows
        #one block per CU for at most 256 columns, its waves walk the tiles of 32 rows
        tiles_m, tiles_n = _cdiv(M, 32), _cdiv(N, 256)
        column_blocks    = _cdiv(_cdiv(N, 32), tiles_n)
        tiles_n          = _cdiv(_cdiv(N, 32), column_blocks)
        blocks, threads, kernel, shared = max(1, min(CONV_SPLIT_ROUND // tiles_n, tiles_m)) * tiles_n, 768, 'conv_gemm_split_short', 0
    params = (_i32(M, N, conv_patch_k(g) if split.patch else K, g.Ho, g.Wo, g.H, g.W, g.Cin, g.KH, g.KW, g.SH, g.SW, g.PH, g.PW, g.DH, g.DW, *g.xs[:3], tiles_m, tiles_n)
              + _u32(flags, *descs, (lhs.size - lhs_offset) * 4, packed.size * 4, (out.size - out_offset) * 4,
                     *_magic_division(g.Ho * g.Wo), *_magic_division(g.Wo))
              + _i32(g.LH, g.LW, g.xs[3], *g.ws, *g.os, split.whole, 0, split.slices, column_blocks if split.short else kpairs // split.slices, kpairs % split.slices))
    derived_ptrs, derived_desc = _conv_derived(epilogue, N)
    operand_slots = _pad([(e.operand, 0) for e in epilogue], CONV_MAX_EPI, (None, 0))
    nbytes = 4 * (lhs.size + packed.size + out.size) + sum(4 * e.operand.size for e in epilogue if e.operand is not None)
    if taps:
        operand_slots[-1] = (taps[0][1], 0)
        nbytes += 4 * taps[0][1].size
    scratch = [(split.partial, 0), (split.arrivals, 0)] if shared else [(None, 0), (None, 0)]
    return Launch(kernel + ('_steps' if steps else ''), (blocks, 1, 1), (threads, 1, 1),
                  [(out, out_offset * 4), (lhs, lhs_offset * 4), (packed, 0)] + scratch + operand_slots + derived_ptrs,
                  params + derived_desc, bytes_moved=nbytes, flops=2 * M * N * K,
                  written=(0, 3, 4) if shared else (0,), scratch=(3, 4) if shared else ())


def conv_product(out: Buffer, lhs: Buffer, rhs: Buffer, g: ConvGeometry, epilogue: tp.Sequence[ConvEpilogueStep] = (), **offsets) -> Launch:
    '''The launch of a product: `rhs` is its packed kernel operand where the geometry carries a plan for the bf16 matrix cores.'''
    return (conv_split_launch if g.split is not None else conv_gemm)(out, lhs, rhs, g, epilogue, **offsets)


def conv_masked_epilogue(epilogue: tp.Sequence[ConvEpilogueStep]) -> tp.Optional[tp.List[tp.Optional[ConvEpilogueStep]]]:
    '''The operands of an epilogue with a mask by their places in the kernel's arguments (full tensor, activation, vector, limit,
    constant; the second result has the last place), or None for one the kernel does not apply.'''
    rest = list(epilogue)
    take = lambda op, kind: rest.pop(0) if rest and rest[0].op == op and rest[0].kind == kind and rest[0].derived is None else None
    full, mask = take(EW['ADD_F'], 3), take(CONV_MASK, 3)
    take(CONV_TAP, 3)
    vector = take(EW['MUL_F'], 2)
    if mask is None or rest:
        return None
    limit, otherwise = (ConvEpilogueStep(EW['NOP'], 1, b) for b in mask.bounds)
    return [full, mask, vector, limit, otherwise]


# --------------------------------------------------------------------------- reductions

RED = dict(reduce_sum=0, reduce_prod=1, reduce_max=2, reduce_min=3, argmax=4, argmin=5)
_RTYPE = {np.dtype('float32'): 0, np.dtype('int32'): 1, np.dtype('uint32'): 2, np.dtype('bool'): 2}


def _pow2_at_least(x: int) -> int:
    p = 1
    while p < x:
        p *= 2
    return p


def _column_block_width(outer: int, R: int, inner: int, nsplit: int) -> int:
    '''Threads side by side along the columns (of four columns each, where their number is a multiple of four) of a block of a column
    reduction. Few blocks with many rows each (the sum of a kernel gradient's slices): narrower blocks, more of them, more
    thread rows walking the rows side by side.'''
    vec = 4 if inner % 4 == 0 else 1
    TI  = min(64, _pow2_at_least(_cdiv(inner, vec)))
    while TI > 8 and 2 * _cdiv(inner, TI * vec) * nsplit * outer <= REDUCE_NARROW_MAX_BLOCKS and _cdiv(R, nsplit) >= 128:
        TI //= 2
    return TI


#Columns of at most this many rows are summed by one launch: a second one costs about 2.3 us. Sums of R x columns in two launches, in one:
#128 x 100 4.6, 2.5 us; 1000 x 10 4.7, 3.2; 1000 x 100 5.1, 3.9; 1536 x 64 5.1, 4.2; 1536 x 1000 5.9, 4.8; 1000 x 9408 9.1, 8.8;
#1536 x 30000 34, 29; 2000 x 100 5.2, 5.4; 4096 x 100 5.3, 8.7. A number of columns that is no multiple of four is read a word at a time,
#and up to eight steps of four rows per thread pay: 1000 x 1001 5.7, 3.7; 512 x 4095 (8 steps) 5.7, 3.6; 1000 x 4095 (16) 6.4, 10.0; 1536 x 1001 (12) 6.0, 6.3;
#512 x 9407 (32) 7.4, 12.7
REDUCE_UNSPLIT_ROWS, REDUCE_UNSPLIT_STEPS = 1536, 8
#Two launches are faster on arrays of some size in two cases (of 368 sums of 256 to 1536 rows and 64 to 80000 columns, one launch always costs 1.5 % more
#than the better of the two on average and up to 25 %, this rule 0.3 % and up to 14). The narrowest blocks read 128 bytes of every row, two lines of memory
#where rows do not begin at a line: 1536 x 4316 7.6 us in two, 9.5 in one, 1536 x 5000 8.4, 9.6, 1400 x 5860 8.8, 10.7, 1100 x 7640 8.8, 10.3; below that
#size 1024 x 5000 (20 MB) 6.8, 6.2, 1536 x 3372 (21) 7.5, 7.6; at whole lines 1536 x 4096 5.8, 4.6. And large arrays for which one launch has too few blocks, as where a
#block more per CU would make them narrower: 900 x 33216 (130 blocks, 120 MB) 20.9, 24.6, 1536 x 36864 (144) 35.1, 39.4; but 1536 x 9408 (147, 58 MB) 12.7, 12.2,
#1536 x 24576 (192) 26.5, 22.7
REDUCE_NARROW_UNSPLIT_BYTES, REDUCE_UNSPLIT_BYTES, REDUCE_UNSPLIT_BLOCKS = 24 << 20, 64 << 20, 160


def _column_sum_starves(outer: int, R: int, inner: int) -> bool:
    '''Whether columns read four at a time are summed faster by two launches although there are few rows.'''
    width, nbytes = _column_block_width(outer, R, inner, 1), 4 * outer * R * inner
    return ((width == 8 and inner % 32 != 0 and nbytes >= REDUCE_NARROW_UNSPLIT_BYTES)
            or (outer * _cdiv(inner, 4 * width) <= REDUCE_UNSPLIT_BLOCKS and nbytes >= REDUCE_UNSPLIT_BYTES))


def plan_reduce_splits(outer: int, R: int, inner: int, op: str, compute_units: int = 256) -> int:
    '''Into how many ranges R is cut so that outer x inner x splits fills the GPU (1 = a single launch).'''
    if op in ('argmax', 'argmin'):
        return 1                                   #index-returning reductions run unsplit
    if inner == 1:
        want  = 32 * compute_units                 #waves
        split = min(_cdiv(want, outer), R // 4096)         #at least 16 KB per wave
    elif R <= REDUCE_UNSPLIT_ROWS and (not _column_sum_starves(outer, R, inner) if inner % 4 == 0 else
                                       _cdiv(R, 4 * (BLOCK // _column_block_width(outer, R, inner, 1))) <= REDUCE_UNSPLIT_STEPS):
        return 1
    else:
        tiles = _cdiv(inner, 256)
        #blocks: several per CU for arrays that stream from HBM for a while; one per CU for smaller ones, whose
        #second launch (it reduces the per-block results) would otherwise take as long as the first
        want  = (4 if outer * R * inner * 4 >= (128 << 20) else 1) * compute_units
        split = min(_cdiv(want, tiles * outer), R // 64)   #at least 64 rows per block
    return max(1, min(split, 65535))


def _reduce_launch(out: Buffer, inp: Buffer, outer: int, R: int, inner: int, op: str, nsplit: int, in_offset_ok=True,
                   prologue: tp.Optional[tp.Tuple[str, tp.Optional[Buffer]]] = None) -> Launch:
    ty   = _RTYPE[inp.dtype]
    mode = {('reduce_sum', 0): 'fsum', ('reduce_max', 0): 'fmax', ('argmax', 0): 'fargmax', ('argmin', 0): 'fargmin'}.get((op, ty), 'any')
    r_chunk = _cdiv(_cdiv(R, nsplit), 4) * 4
    nsplit  = _cdiv(R, r_chunk)
    if inner == 1:
        vec = 4 if R % 4 == 0 else 1
        params = _u32(outer, R, 1, RED[op], ty, r_chunk, nsplit, 0)
        return Launch(f'reduce_rows_{mode}_v{vec}', (_cdiv(outer * nsplit, 4), 1, 1), (BLOCK, 1, 1), [(out, 0), (inp, 0)], params,
                      bytes_moved=4 * (outer * R + outer * nsplit)), nsplit
    vec = 4 if inner % 4 == 0 else 1
    TI  = _column_block_width(outer, R, inner, nsplit)
    params = _u32(outer, R, inner, RED[op], ty, r_chunk, nsplit, TI)
    blocks = _cdiv(inner, TI * vec) * nsplit * outer
    if blocks >= 2**31:
        raise NotImplementedError(f'reduction with {outer} outer rows and inner size {inner}')
    if prologue is not None:
        #the operand's element-wise producer applied while loading: ('mul', array of the same shape),
        #('mulv', vector over inner) or ('neg', None); float column sums only
        kind, second = prologue
        assert mode == 'fsum' and kind in ('mul', 'mulv', 'neg') and (second is None) == (kind == 'neg')
        assert second is None or second.size == (outer * R * inner if kind == 'mul' else inner)
        extra = 0 if second is None else second.size
        return Launch(f'reduce_cols_fsum_{kind}_v{vec}', (blocks, 1, 1), (BLOCK, 1, 1), [(out, 0), (inp, 0), (second, 0)], params,
                      bytes_moved=4 * (outer * R * inner + outer * nsplit * inner + extra)), nsplit
    return Launch(f'reduce_cols_{mode}_v{vec}', (blocks, 1, 1), (BLOCK, 1, 1), [(out, 0), (inp, 0)], params,
                  bytes_moved=4 * (outer * R * inner + outer * nsplit * inner)), nsplit


def reduce(out: Buffer, inp: Buffer, outer: int, R: int, inner: int, op: str,
           partial: tp.Optional[Buffer] = None, nsplit: int = 1, prologue=None) -> tp.List[Launch]:
    '''[outer, R, inner] -> [outer, inner]. With nsplit > 1, `partial` (outer * nsplit * inner words) receives
    the per-range results of a first launch and a second launch reduces them. `prologue`: see _reduce_launch.'''
    if nsplit <= 1:
        return [_reduce_launch(out, inp, outer, R, inner, op, 1, prologue=prologue)[0]]
    first, nsplit = _reduce_launch(partial, inp, outer, R, inner, op, nsplit, prologue=prologue)
    if nsplit == 1:
        return [_reduce_launch(out, inp, outer, R, inner, op, 1, prologue=prologue)[0]]
    assert partial.size >= outer * nsplit * inner and partial.dtype == inp.dtype
    second = _reduce_launch(out, partial, outer, nsplit, inner, op, 1)[0]
    return [first, second]


def column_sum_update(column_sum: Launch, out: Buffer, minuend: Buffer, rate: Buffer) -> tp.Optional[Launch]:
    '''out = minuend - rate * (what `column_sum` writes), in the order of its additions; None where `column_sum` is not an
    unsplit float column sum of one [R, inner] array.'''
    if column_sum.kernel not in REDUCE_BATCH_KERNELS:
        return None
    outer, R, inner, _, _, _, nsplit, TI = (int(v) for v in np.frombuffer(column_sum.params, dtype=np.uint32))
    if (outer, nsplit) != (1, 1):
        return None
    assert out.size == minuend.size == inner and rate.size == 1
    return Launch(column_sum.kernel.replace('fsum_', 'fsum_update_'), column_sum.grid, column_sum.block,
                  [(out, 0), column_sum.buffers[1], (minuend, 0), (rate, 0)], _u32(R, inner, TI), bytes_moved=column_sum.bytes_moved + 4 * inner)


def scale_relu_backward(column_sum: Launch, dx: Buffer, sum_m: Buffer, sum_mx: Buffer, x: Buffer, scale: Buffer, cotangent: Buffer,
                        select: tp.Optional[tp.Tuple[Buffer, Buffer, Buffer]] = None) -> Launch:
    '''dx = m * scale (scale a vector over the columns), and sum_m, sum_mx receive what `column_sum`, a reduce_cols
    launch over an array of that shape, would write for m and for m * x (same grid, same parameters, same order
    of additions). m is the cotangent itself, or with select = (ans, threshold, otherwise), two single values:
    ans > threshold ? cotangent : otherwise.'''
    assert column_sum.kernel in ('reduce_cols_fsum_v1', 'reduce_cols_fsum_v4'), column_sum.kernel
    n = cotangent.size
    assert dx.size == x.size == n
    ans, threshold, otherwise = select if select is not None else (None, None, None)
    assert select is None or (ans.size == n and threshold.size == otherwise.size == 1)
    name = 'scale_relu_backward_' if select is not None else 'scale_backward_'
    return Launch(name + column_sum.kernel[-2:], column_sum.grid, column_sum.block,
                  [(dx, 0), (sum_m, 0), (sum_mx, 0), (ans, 0), (threshold, 0), (cotangent, 0), (otherwise, 0), (x, 0), (scale, 0)],
                  column_sum.params, bytes_moved=4 * ((4 if select is not None else 3) * n + 2 * scale.size), written=(0, 1, 2))


def relu_backward(column_sum: Launch, m: Buffer, sum_m: Buffer, cotangent: Buffer, select: tp.Tuple[Buffer, Buffer, Buffer]) -> Launch:
    '''m = ans > threshold ? cotangent : otherwise with select = (ans, threshold, otherwise), and sum_m receives what
    `column_sum` would write for m.'''
    assert column_sum.kernel in REDUCE_BATCH_KERNELS, column_sum.kernel
    ans, threshold, otherwise = select
    assert ans.size == cotangent.size == m.size and threshold.size == otherwise.size == 1
    return Launch('relu_backward_' + column_sum.kernel[-2:], column_sum.grid, column_sum.block,
                  [(m, 0), (sum_m, 0), (ans, 0), (threshold, 0), (cotangent, 0), (otherwise, 0)], column_sum.params,
                  bytes_moved=12 * m.size + 4 * sum_m.size, written=(0, 1))


def sum_with_post(total: Launch, out: Buffer, kind: str, value: Buffer) -> tp.Optional[Launch]:
    '''An unsplit float sum that stores sum / value, sum * value or -(sum / value) (kind 'div', 'times', 'negdiv'; one value).'''
    if total.kernel not in ('reduce_rows_fsum_v1', 'reduce_rows_fsum_v4') + REDUCE_BATCH_KERNELS:
        return None
    if np.frombuffer(total.params, dtype=np.uint32)[6] != 1:
        return None
    assert kind in ('div', 'times', 'negdiv') and value.size == 1 and out.size == total.buffers[0][0].size
    return Launch(total.kernel.replace('fsum_', f'fsum_{kind}_'), total.grid, total.block, [(out, 0), total.buffers[1], (value, 0)], total.params,
                  bytes_moved=total.bytes_moved)


SOFTMAX_MAX_ROW = 4096      #rows this short run unsplit in reduce_rows, whose summation order softmax_rows repeats
#vectors per lane of the kernels' variants: a row stays in the registers of one wave
SOFTMAX_VECTORS = {4: (1, 2, 3, 4, 6, 8, 12, 16), 1: (1, 2, 3, 4, 6, 8, 12, 16, 24, 32, 48, 64)}


def softmax_rows(out: Buffer, inp: Buffer, outer: int, R: int, arg_out: tp.Optional[Buffer] = None) -> Launch:
    '''exp(x - max) / sum(exp(x - max)) over the rows of [outer, R]; see softmax_rows_body in reduce.hip.
    `arg_out`: also the arg-max of every result row (int32 [outer]).'''
    assert 0 < R < SOFTMAX_MAX_ROW and inp.size == out.size == outer * R and (arg_out is None or arg_out.size == outer)
    vec     = 4 if R % 4 == 0 else 1
    vectors = next(n for n in SOFTMAX_VECTORS[vec] if n * 64 * vec >= R)
    #short rows share a wave: as few lanes each as hold them
    lanes   = _pow2_at_least(R // vec) if vectors == 1 else 64
    kernel  = f'softmax_rows_v{vec}' + (f'_n{vectors}' if vectors > 1 else '')
    return Launch(kernel, (_cdiv(outer, 4 * (64 // lanes)), 1, 1), (BLOCK, 1, 1), [(out, 0), (inp, 0), (arg_out, 0)],
                  _u32(outer, R, lanes.bit_length() - 1), bytes_moved=8 * outer * R + (4 * outer if arg_out is not None else 0),
                  streamable=True, written=(0, 2))


# ---------------------------------------------------------------- row programs (rows.hip)

ROWS_MAX_IN, ROWS_MAX_OUT, ROWS_MAX_CODE = 8, 6, 48
ROWS_OPS     = dict(load=0, apply=1, reduce_sum=2, reduce_max=3, put=4, out=5)
ROWS_MAX_ROW = 1024                 #a row stays in the registers of one wave, 16 values per lane
#(values per vector, vectors per lane) of the kernels' variants
ROWS_VARIANTS = ((4, 1), (4, 4), (1, 1), (1, 4), (1, 16))
ROWS_LDS     = 64 << 10


class RowsInput(tp.NamedTuple):
    '''An array a row program reads: element base + row * row_stride + column * column_stride; `single`: one value per row.'''
    buffer:        Buffer
    base:          int
    row_stride:    int
    column_stride: int
    single:        bool


class RowsStep(tp.NamedTuple):
    '''One instruction: `slot` is a pair (kind, number) - ('in', input), ('value', number of a value put away) or
    ('out', output) - or None; `single`: one value per row.'''
    what:   str
    op:     int = 0
    left:   bool = False
    slot:   tp.Optional[tp.Tuple[str, int]] = None
    single: bool = False
    imm:    int = 0


def rows_variant(R: int) -> tp.Tuple[int, int]:
    '''The order of additions is that of reduce_rows: 16-byte vectors where the row has a multiple of 4 values.'''
    vec = 4 if R % 4 == 0 else 1
    return vec, next(n for v, n in ROWS_VARIANTS if v == vec and 64 * v * n >= R)


def _rows_slots(steps: tp.Sequence[RowsStep], inputs: tp.Sequence[RowsInput], width: int) -> tp.Tuple[tp.Dict, int]:
    '''First word of every slot and the number of words: a slot is handed on once what it holds is not read any more.'''
    sizes, last = {('in', k): 1 if i.single else width for k, i in enumerate(inputs)}, {}
    for at, s in enumerate(steps):
        if s.slot is not None and s.slot[0] != 'out':
            sizes.setdefault(s.slot, 1 if s.single else width)
            last[s.slot] = at
    place, free, words = {}, {1: [], width: []}, 0

    def give(slot):
        nonlocal words
        n = sizes[slot]
        if free[n]:
            place[slot] = free[n].pop()
        else:
            place[slot] = words
            words += n

    for k in range(len(inputs)):
        give(('in', k))
    for at, s in enumerate(steps):
        if s.what == 'put':
            give(s.slot)
        for slot in [x for x, end in last.items() if end == at]:
            free[sizes[slot]].append(place[slot])
    return place, words


def row_program(outs: tp.Sequence[Buffer], inputs: tp.Sequence[RowsInput], steps: tp.Sequence[RowsStep], outer: int, R: int) -> tp.Optional[Launch]:
    '''One launch for element-wise steps and reductions over the rows of [outer, R]; see rows.hip. None where the program
    does not fit the kernel.'''
    vec, vectors = rows_variant(R)
    place, words = _rows_slots(steps, inputs, vec * vectors)
    waves = next((w for w in (4, 2, 1) if words * 4 * 64 * w <= ROWS_LDS), None)
    if waves is None or len(inputs) > ROWS_MAX_IN or len(outs) > ROWS_MAX_OUT or len(steps) > ROWS_MAX_CODE:
        return None
    lanes = min(64, _pow2_at_least(R // vec)) if vectors == 1 else 64
    flags = [place['in', k] | (i.single << 16)
             | ((vec == 4 and i.column_stride == 1 and i.row_stride % 4 == 0 and i.base % 4 == 0) << 17) for k, i in enumerate(inputs)]
    code, one_value = [], False                 #one_value: the accumulator is the same in all columns of a row
    for s in steps:
        slot = 0 if s.slot is None else s.slot[1] if s.slot[0] == 'out' else place[s.slot]
        once = s.what == 'apply' and one_value and (s.slot is None or s.single)
        code += [ROWS_OPS[s.what] | s.op << 4 | bool(s.left) << 16 | bool(s.single) << 17 | (s.slot is not None) << 18 | once << 19 | slot << 20, s.imm]
        one_value = {'apply': once, 'load': bool(s.single), 'put': one_value, 'out': one_value}.get(s.what, True)
    params = (_u32(outer, R, lanes.bit_length() - 1 | 64 * waves << 8, len(inputs), len(steps), *_pad([i.buffer.size * 4 for i in inputs], ROWS_MAX_IN),
                   *_pad([i.base for i in inputs], ROWS_MAX_IN))
              + _i32(*_pad([i.row_stride for i in inputs], ROWS_MAX_IN), *_pad([i.column_stride for i in inputs], ROWS_MAX_IN))
              + _u32(*_pad(flags, ROWS_MAX_IN), *_pad(code, 2 * ROWS_MAX_CODE)))
    nbytes = sum(4 * min(b.size, outer * R) for b in [i.buffer for i in inputs] + list(outs))
    return Launch(f'rows_v{vec}_n{vectors}', (_cdiv(outer, waves * (64 // lanes)), 1, 1), (64 * waves, 1, 1),
                  _pad([(b, 0) for b in outs], ROWS_MAX_OUT, (None, 0)) + _pad([(i.buffer, 0) for i in inputs], ROWS_MAX_IN, (None, 0)),
                  params, lds=4 * words * 64 * waves, bytes_moved=nbytes, written=tuple(range(len(outs))))


def reduce_general(out: Buffer, inp: Buffer, kept, reduced, op: str) -> Launch:
    '''kept / reduced: lists of (size, stride) in row-major order of the output / of the reduce index.'''
    if len(kept) > 4 or len(reduced) > 4:
        raise NotImplementedError('reduction over more than 4 separate dimension groups')
    n_out = int(np.prod([k[0] for k in kept], dtype=np.int64))
    n_red = int(np.prod([r[0] for r in reduced], dtype=np.int64))
    params = _u32(n_out, n_red, RED[op], _RTYPE[inp.dtype], len(kept), len(reduced),
                  *_pad([k[0] for k in kept], 4, 1), *_pad([k[1] for k in kept], 4),
                  *_pad([r[0] for r in reduced], 4, 1), *_pad([r[1] for r in reduced], 4))
    return Launch('reduce_general', (_cdiv(n_out, 4), 1, 1), (BLOCK, 1, 1), [(out, 0), (inp, 0)], params,
                  bytes_moved=4 * (inp.size + out.size))


def _pool_divisions(dims) -> bytes:
    '''PoolParams.div_magic / div_shift for an array [batch, height, width, channels]: channels, width, height.'''
    pairs = [_magic_division(d) for d in (dims[3], dims[2], dims[1])]
    return _u32(*[m for m, _ in pairs], *[sh for _, sh in pairs])


def pool(out: Buffer, inp: Buffer, op: str, window, strides, pad_low, dilation) -> Launch:
    rank = len(inp.shape)
    if rank > 4:
        raise NotImplementedError('window reductions over more than 4 dimensions')
    lead     = 4 - rank
    in_dims  = [1] * lead + list(inp.shape)
    out_dims = [1] * lead + list(out.shape)
    window   = [1] * lead + list(window)
    strides  = [1] * lead + list(strides)
    dilation = [1] * lead + list(dilation)
    pad_low  = [0] * lead + list(pad_low)
    n   = out.size
    vec = 4 if (window[3] == 1 and strides[3] == 1 and pad_low[3] == 0 and in_dims[3] % 4 == 0
                and in_dims[3] == out_dims[3]) else 1
    params = (_u32(n, RED[op], _RTYPE[inp.dtype], *in_dims, *out_dims, *window, *strides, *dilation) + _i32(*pad_low)
              + _pool_divisions(out_dims))
    #[batch, y, x, channels] with a 3x3 or 2x2 window over y and x: the kernel that requests all taps at once
    if (vec == 4 and window[0] == 1 and strides[0] == 1 and pad_low[0] == 0 and in_dims[0] == out_dims[0]
            and (window[1], window[2]) in ((3, 3), (2, 2)) and inp.size * 4 < 2**31 and n * 4 < 2**32):
        return Launch(f'pool2d_{window[1]}x{window[2]}_v4', (_cdiv(_cdiv(n, 4), BLOCK), 1, 1), (BLOCK, 1, 1), [(out, 0), (inp, 0)], params,
                      bytes_moved=4 * (inp.size + out.size))
    return Launch(f'pool_v{vec}', (_cdiv(_cdiv(n, vec), BLOCK), 1, 1), (BLOCK, 1, 1), [(out, 0), (inp, 0)], params,
                  bytes_moved=4 * (inp.size + out.size))


POOL_SUM_STEPS = {'div': 1, 'times': 2, 'select': 3}


def pool_sum(out: Buffer, source: EwOperand, source_extent, low, spread, window, strides, dilation, before=None, after=None) -> tp.Optional[Launch]:
    '''Float sums under windows over y and x of [batch, y, x, channels], out = after(sum(before(source) on a grid of zeros)); None where the kernel
    does not apply. `source` reads [batch, *source_extent, channels] through its strides; its elements lie `spread` apart behind `low`
    zeros (a negative number cuts none off: the padding of the windows). `before`, `after`: None, ('div' | 'times', one value), and
    for `after` ('select', threshold, otherwise, compared array): compared > threshold ? sum : otherwise.'''
    if len(out.shape) != 4 or tuple(window) not in ((3, 3), (2, 2)) or out.size == 0:
        return None
    batch, Ho, Wo, C = out.shape
    sb, sy, sx, sc = source.strides
    if (C % 4 or sc != 1 or source.offset % 4 or any(st % 4 or st < 0 for st in (sb, sy, sx)) or source.buffer.size * 4 >= 2**31 or out.size * 4 >= 2**31
            or min(spread) < 1 or max(*spread, *strides, *dilation, *source_extent, Ho, Wo, abs(low[0]), abs(low[1])) >= 1 << 14):
        return None
    words = source.buffer.size - source.offset
    params = (_u32(out.size, Ho, Wo, C, *source_extent, sb, sy, sx, words) + _i32(-low[0], -low[1]) + _u32(*strides, *dilation, *spread,
              POOL_SUM_STEPS[before[0]] if before else 0, POOL_SUM_STEPS[after[0]] if after else 0) + _pool_divisions(out.shape))
    compared = otherwise = None
    if after is not None and after[0] == 'select':
        otherwise, compared = after[2:]
        assert compared.size == out.size
    buffers = [(out, 0), (source.buffer, source.offset * 4)] + [(b, 0) for b in (before[1] if before else None, after[1] if after else None, compared, otherwise)]
    spreading = 'pad_nd_' if tuple(spread) != (1, 1) else ''
    return Launch(f'{spreading}pool2d_sum_{window[0]}x{window[1]}_v4', (_cdiv(out.size // 4, BLOCK), 1, 1), (BLOCK, 1, 1), buffers, params,
                  bytes_moved=4 * (min(source.buffer.size, batch * int(np.prod(source_extent)) * C) + out.size * (2 if compared is not None else 1)))


def select_scatter_add(out: Buffer, source: Buffer, operand: Buffer, selected: Buffer, op: str, window, strides, pad_low) -> tp.List[Launch]:
    '''Gradient of a max (`op` = 'reduce_max': select with ge) or min pooling in two launches: the selected tap
    of every window into `selected` (uint32, source's shape), then the per-element sums; see reduce.hip.'''
    rank = len(operand.shape)
    if rank > 4:
        raise NotImplementedError('select_and_scatter_add over more than 4 dimensions')
    lead     = 4 - rank
    in_dims  = [1] * lead + list(operand.shape)
    out_dims = [1] * lead + list(source.shape)
    window   = [1] * lead + list(window)
    strides  = [1] * lead + list(strides)
    pad_low  = [0] * lead + list(pad_low)
    vec = 4 if (window[3] == 1 and strides[3] == 1 and pad_low[3] == 0 and in_dims[3] % 4 == 0
                and in_dims[3] == out_dims[3]) else 1
    if max(in_dims) >= 2**31 or any(abs(p) >= 2**30 for p in pad_low):
        raise NotImplementedError('select_and_scatter_add: dimension too large')
    assert tuple(selected.shape) == tuple(source.shape) and selected.dtype == np.uint32
    tail = _u32(RED[op], _RTYPE[operand.dtype], *in_dims, *out_dims, *window, *strides, 1, 1, 1, 1) + _i32(*pad_low)
    n_win, n = source.size, operand.size
    select, scatter = f'select_window_v{vec}', f'scatter_selected_v{vec}'
    #[batch, y, x, channels] floats with a 3x3 or 2x2 window over y and x: the kernels that request everything at once
    if (vec == 4 and window[0] == 1 and strides[0] == 1 and pad_low[0] == 0 and in_dims[0] == out_dims[0] and CHOICES.pool_gradient_2d is not False
            and (window[1], window[2]) in ((3, 3), (2, 2)) and operand.dtype == np.float32 and n * 4 < 2**31 and n_win * 4 < 2**31):
        #(an element lies in at most ceil(window / stride) windows per dimension; the variants are square in that count)
        most = max(_cdiv(window[1], strides[1]), _cdiv(window[2], strides[2]))
        select, scatter = f'select_window2d_{window[1]}x{window[2]}_v4', f'scatter_selected2d_{window[1]}x{window[2]}_n{most}x{most}_v4'
    first  = Launch(select, (_cdiv(_cdiv(n_win, vec), BLOCK), 1, 1), (BLOCK, 1, 1),
                    [(selected, 0), (operand, 0)], _u32(n_win) + tail + _pool_divisions(out_dims), bytes_moved=4 * (operand.size + source.size))
    second = Launch(scatter, (_cdiv(_cdiv(n, vec), BLOCK), 1, 1), (BLOCK, 1, 1),
                    [(out, 0), (source, 0), (selected, 0)], _u32(n) + tail + _pool_divisions(in_dims), bytes_moved=4 * (operand.size + 2 * source.size),
                    streamable=vec == 4 and n < 2**31)
    #3 x 3 windows at a stride of 2: a thread per group of 2 x 2 elements (by four channels), which shares its windows' loads
    if ('2d_3x3' in scatter and (strides[1], strides[2]) == (2, 2) and 0 <= pad_low[1] < 3 and 0 <= pad_low[2] < 3
            and CHOICES.pool_gradient_2d != 'elements'):
        groups = [((extent + pad - 1) >> 1) - (pad >> 1) + 1 for extent, pad in ((in_dims[1], pad_low[1]), (in_dims[2], pad_low[2]))]
        n_groups = in_dims[0] * groups[0] * groups[1] * in_dims[3]
        second = second._replace(kernel='scatter_selected2d_3x3_s2_v4', grid=(_cdiv(_cdiv(n_groups, 4), BLOCK), 1, 1),
                                 params=_u32(n_groups) + tail + _pool_divisions([in_dims[0], groups[0], groups[1], in_dims[3]]),
                                 streamable=n_groups < 2**31)
    return [first, second]


PAD_MAX_RANK = 6


def _merged_pad_dims(out_shape, in_shape, padding_config):
    '''(out extent, in extent, low, step) per dimension after folding every dimension the padding leaves alone into
    the one before it when that one has no interior padding: (w, c) -> w * C + c turns `low` into low * C.'''
    dims = [(int(o), int(i), int(c[0]), int(c[2]) + 1) for o, i, c in zip(out_shape, in_shape, padding_config)]
    merged: tp.List[tp.Tuple[int, int, int, int]] = []
    for o, i, low, step in reversed(dims):
        if merged:
            o2, i2, low2, step2 = merged[-1]
            if low2 == 0 and step2 == 1 and o2 == i2 and step == 1:
                merged[-1] = (o * o2, i * o2, low * o2, 1)
                continue
        merged.append((o, i, low, step))
    return merged[::-1]


def pad(out: Buffer, inp: Buffer, value: Buffer, padding_config) -> Launch:
    dims = _merged_pad_dims(out.shape, inp.shape, padding_config)
    if len(dims) > PAD_MAX_RANK:
        raise NotImplementedError('pad with rank > 6')
    if max(out.size, inp.size) >= 2**32 - 2**12 or any(abs(d[2]) >= 2**31 for d in dims):
        raise NotImplementedError('pad of arrays with 2^32 elements or more')
    #the dimensions fill the front of the tables (the kernel does not split its index for dimension 0) and the unused
    #ones behind them have extent 1; an empty operand keeps an extent of 0 no index can fall into
    dims = dims + [(1, 1, 0, 1)] * (PAD_MAX_RANK - len(dims))
    last = max((d for d in range(PAD_MAX_RANK) if dims[d][:3] != (1, 1, 0)), default=0)
    o, i, low, step = dims[last]
    vec = 4 if (step == 1 and low % 4 == 0 and o % 4 == 0 and i % 4 == 0) else 1
    params = _u32(out.size, *[d[0] for d in dims], *[d[1] for d in dims]) + _i32(*[d[2] for d in dims]) + _u32(*[d[3] for d in dims])
    return Launch(f'pad_nd_v{vec}', (_cdiv(_cdiv(out.size, vec), BLOCK), 1, 1), (BLOCK, 1, 1),
                  [(out, 0), (inp, 0), (value, 0)], params, bytes_moved=4 * (inp.size + out.size), streamable=vec == 4 and out.size < 2**31)


# --------------------------------------------------------------------------- gather / scatter / rng

IDX_MAX_RANK = 6


def gather_rows(out: Buffer, table: Buffer, idx: Buffer, n_idx: int, row_len: int, n_rows: int, idx_stride: int = 1,
                fill: tp.Optional[int] = None) -> Launch:
    '''`fill`: None clamps rows outside the table; a 32-bit pattern makes them read as that value instead.'''
    vec = 4 if row_len % 4 == 0 else 1
    total = n_idx * (row_len // vec)
    return Launch(f'gather_rows_v{vec}', (_cdiv(total, BLOCK), 1, 1), (BLOCK, 1, 1), [(out, 0), (table, 0), (idx, 0)],
                  _u32(n_idx, row_len, n_rows, idx_stride, int(fill is not None), fill or 0, 0), bytes_moved=4 * (2 * n_idx * row_len + n_idx),
                  streamable=vec == 4 and n_idx < 2**31)


def gather_general(out: Buffer, operand: Buffer, indices: Buffer, offset_dims, collapsed, start_index_map, slice_sizes,
                   fill: tp.Optional[int] = None) -> Launch:
    out_rank, op_rank = len(out.shape), len(operand.shape)
    if max(out_rank, op_rank, len(indices.shape)) > IDX_MAX_RANK:
        raise NotImplementedError('gather with rank > 6')
    batch_dims = list(indices.shape[:-1])
    params = _u32(out.size, out_rank, op_rank, indices.shape[-1],
                  *_pad(out.shape, IDX_MAX_RANK, 1), *_pad([int(d in offset_dims) for d in range(out_rank)], IDX_MAX_RANK),
                  *_pad(operand.shape, IDX_MAX_RANK, 1), *_pad(row_major_strides(operand.shape), IDX_MAX_RANK),
                  *_pad(slice_sizes, IDX_MAX_RANK, 1), *_pad([int(d in collapsed) for d in range(op_rank)], IDX_MAX_RANK),
                  *_pad(start_index_map, IDX_MAX_RANK), *_pad(batch_dims, IDX_MAX_RANK, 1), len(batch_dims),
                  int(fill is not None), fill or 0)
    return Launch('gather_general', (_cdiv(out.size, BLOCK), 1, 1), (BLOCK, 1, 1), [(out, 0), (operand, 0), (indices, 0)],
                  params, bytes_moved=4 * (2 * out.size + indices.size))


#kernels that can add a value to negative indices themselves: position of the index array among their arguments, and the
#byte offset of the `wrap` field in their parameter block
INDEX_WRAP_KERNELS = {'gather_rows_v1': (2, 24), 'gather_rows_v4': (2, 24), 'scatter_rows_rank': (3, 24)}


def with_wrapped_index(launch: Launch, raw: Buffer, raw_byte_offset: int, amount: int) -> Launch:
    '''`launch` reading the raw index array `raw` instead of its normalised copy, adding `amount` to negative indices itself.'''
    position, field = INDEX_WRAP_KERNELS[launch.kernel]
    assert launch.params[field:field + 4] == _u32(0)
    buffers = list(launch.buffers)
    buffers[position] = (raw, buffers[position][1] + raw_byte_offset)
    return launch._replace(buffers=buffers, params=launch.params[:field] + _u32(amount) + launch.params[field + 4:])


def scatter_add_rows(out: Buffer, idx: Buffer, updates: Buffer, n_idx: int, row_len: int, n_rows: int, idx_stride: int = 1,
                     clip: bool = False) -> Launch:
    '''`clip`: rows outside the table go to its first / last row instead of being dropped.'''
    total = n_idx * row_len
    return Launch('scatter_add_rows', (_cdiv(total, BLOCK), 1, 1), (BLOCK, 1, 1), [(out, 0), (idx, 0), (updates, 0)],
                  _u32(n_idx, row_len, n_rows, idx_stride, int(out.dtype == np.float32), int(clip)),
                  bytes_moved=4 * (total + n_idx + out.size))


SCATTER_MAX_CAP = 1024


def choose_scatter_bucket_cap(n_idx: int, n_rows: int, row_len: int) -> int:
    '''How many slots every table row gets in the sorted scatter-add's table of fixed-capacity buckets (0: none, every
    update goes through the overflow table): four times the average number of updates per row, as a power of two
    between 8 and 1024 - with indices spread evenly a row with more than that is a rarity - as long as the slots take at
    most eight words per update, or 64 MB. Updates beyond the slots cost a hash table's insertion and a search each (rows x row length,
    updates: us of gather and scatter-add with 0, 8, 16, 32, 64, 128, 256 slots): 100000 x 16, 262144 1104, 65, 64, 64, 64, 64, 64; 20000 x 16, 262144
    427, 259, 76, 42, 42, 42, 42; 100000 x 24, 32000 330, 30, 30, 30, 30, 30, 31; 5000 x 200, 90000 116, 109, 81, 42, 41, 41, 41; 1000 x 256,
    262144 5340, 4496, 3724, 2440, 685, 199, 194; 65536 x 256, 262144 869, 150, 148, 148, 148, 148, 148.'''
    if CHOICES.scatter_bucket_cap is not None:
        cap = int(CHOICES.scatter_bucket_cap)
        assert 0 <= cap <= SCATTER_MAX_CAP
        return cap
    if n_rows == 0 or n_idx == 0:
        return 0
    cap = 8
    while cap < SCATTER_MAX_CAP and cap * n_rows < 4 * n_idx:
        cap *= 2
    while cap >= 4 and cap * n_rows > max(8 * n_idx, 1 << 24):
        cap //= 2
    return cap if cap >= 4 else 0


def scatter_table_slots(n_idx: int) -> int:
    '''Slots of the overflow table of a sorted scatter-add of n_idx updates: a power of two, at least 64 and at least
    twice the number of updates.'''
    return max(64, _pow2_at_least(2 * n_idx))


def scatter_add_rows_sorted(out: Buffer, operand: Buffer, idx: Buffer, updates: Buffer, count: Buffer, table: Buffer, gathered: Buffer,
                            sorted_: Buffer, n_idx: int, row_len: int, n_rows: int, operand_is_scalar: bool = False,
                            idx_stride: int = 1, clip: bool = False, fixed: tp.Optional[Buffer] = None, cap: int = 0) -> tp.List[Launch]:
    '''out = operand; out[idx[i], :] += updates[i, :] without atomics on the data: the first launch buckets the updates by
    row, then one wave per row, or for several short ones, sums their buckets. `count`: n_rows + 1 words, `table`: two words per slot of the overflow
    table (scatter_table_slots), both zero before and after; `fixed`: n_rows * cap words, the first `cap` updates of
    every row (cap = 0: no such table); `gathered`, `sorted_`: n_idx words each, room for the buckets of rows with
    more than cap updates. `operand` is the table, or one word when the table is a constant filled with a single
    value.'''
    slots = scatter_table_slots(n_idx)
    assert count.size == n_rows + 1 and table.size == 2 * slots and gathered.size == n_idx and sorted_.size == n_idx
    assert 0 <= cap <= SCATTER_MAX_CAP and (cap == 0 or (fixed is not None and fixed.size == n_rows * cap))
    if fixed is None:
        fixed = gathered                 #(never touched: no update's number within its row is below 0)
    params = _u32(n_idx, row_len, n_rows, idx_stride, int(operand_is_scalar), int(clip), 0, cap, slots - 1)
    vec    = 4 if row_len % 4 == 0 else 1
    kind   = 'f' if out.dtype == np.float32 else 'i'
    table_passes = 1 if operand_is_scalar else 2
    lanes = max(4, _pow2_at_least(row_len // vec))
    #Several rows per wave where there are more rows than waves the chip holds and few updates for each (us of gather and scatter-add, one row per
    #wave and several; rows x row length, updates: 100000 x 16, 262144 64.5, 39.9; 100000 x 24, 32000 30.7, 17.5; 20000 x 24, 100000 25.8, 20.8; 40000 x 31, 131072 40.4, 36.6;
    #but 5000 x 24, 32000 12.8, 15.2; 12000 x 40, 96000 25.4, 28.8; 20000 x 16, 262144 42.3, 65.9; 30000 x 128, 60000 32.6, 33.4)
    short = (cap >= 8 and lanes <= 32 and
             (CHOICES.scatter_short_rows if CHOICES.scatter_short_rows is not None else row_len <= 64 and n_rows >= 8192 and n_idx <= 6 * n_rows))
    return [
        Launch('scatter_rows_rank', (_cdiv(n_idx, BLOCK), 1, 1), (BLOCK, 1, 1), [(count, 0), (fixed, 0), (table, 0), (idx, 0)], params,
               bytes_moved=8 * n_idx, written=(0, 1, 2)),
        Launch(f'scatter_rows_sum_{"short_" if short else ""}{kind}_v{vec}', (_cdiv(n_rows, 4 * (64 // lanes if short else 1)), 1, 1), (BLOCK, 1, 1),
               [(out, 0), (operand, 0), (updates, 0), (count, 0), (fixed, 0), (table, 0), (gathered, 0), (sorted_, 0)],
               params + (_u32(lanes.bit_length() - 1) if short else b''),
               bytes_moved=4 * (n_idx * row_len + n_idx + n_rows + table_passes * n_rows * row_len), written=(0, 3, 5, 6, 7)),
    ]


def scatter_add_general(out: Buffer, indices: Buffer, updates: Buffer, update_window_dims, inserted_window_dims,
                        scatter_dims_to_operand_dims, clip: bool = False) -> Launch:
    upd_rank, op_rank = len(updates.shape), len(out.shape)
    if max(upd_rank, op_rank, len(indices.shape)) > IDX_MAX_RANK:
        raise NotImplementedError('scatter-add with rank > 6')
    window_dims = [updates.shape[d] for d in update_window_dims]
    it = iter(window_dims)
    window_sizes = [1 if d in inserted_window_dims else next(it) for d in range(op_rank)]
    batch_dims = list(indices.shape[:-1])
    params = _u32(updates.size, upd_rank, op_rank, indices.shape[-1], int(out.dtype == np.float32),
                  *_pad(updates.shape, IDX_MAX_RANK, 1), *_pad([int(d in update_window_dims) for d in range(upd_rank)], IDX_MAX_RANK),
                  *_pad(out.shape, IDX_MAX_RANK, 1), *_pad(row_major_strides(out.shape), IDX_MAX_RANK),
                  *_pad([int(d in inserted_window_dims) for d in range(op_rank)], IDX_MAX_RANK),
                  *_pad(window_sizes, IDX_MAX_RANK, 1), *_pad(scatter_dims_to_operand_dims, IDX_MAX_RANK),
                  *_pad(batch_dims, IDX_MAX_RANK, 1), int(clip))
    return Launch('scatter_add_general', (_cdiv(max(updates.size, 1), BLOCK), 1, 1), (BLOCK, 1, 1),
                  [(out, 0), (indices, 0), (updates, 0)], params, bytes_moved=4 * (updates.size + indices.size + out.size))


def threefry2x32(out0: Buffer, out1: Buffer, key0: Buffer, key1: Buffer, x0: Buffer, x1: Buffer, key_is_scalar: bool) -> Launch:
    n   = x0.size
    vec = 4 if n % 4 == 0 else 1
    return Launch(f'threefry2x32{"_k" if key_is_scalar else ""}_v{vec}', (_cdiv(_cdiv(n, vec), BLOCK), 1, 1), (BLOCK, 1, 1),
                  [(out0, 0), (out1, 0), (key0, 0), (key1, 0), (x0, 0), (x1, 0)], _u32(n, int(key_is_scalar)),
                  bytes_moved=16 * n, written=(0, 1))
