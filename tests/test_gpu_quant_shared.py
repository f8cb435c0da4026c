"""Workgroups that share their groups (`quant_shared_kernel`): rows that do not fill the last workgroup or step, more rows than the
registers hold, octets that are no power of two, kept inner indices that do not fill the last tile, groups of whole rows; with the
others' extremes waited for and, without waiting, with their rows read by whoever comes first.  Bit-exact against the CPU oracle."""
import math

import pytest
import torch

import varq_oracle as O
from gpu_util import note
from test_gpu_nonfinite import WHAT, _bits, _spoil
from var_q_amd import _lib, ops

pytestmark = pytest.mark.gpu


DTYPE = {torch.float32: 0, torch.bfloat16: 1, torch.float16: 2}


def _shards(x, dims, word_bits, asym, tensors=1):
    return _shards_of(x.shape, x.dtype, dims, word_bits, asym, tensors)


def _shards_of(shape, dtype, dims, word_bits, asym, tensors=1):
    """Workgroups that share each group; 1: one workgroup by itself, 0: the input is read twice."""
    return _lib.load().varq_quant_pack_shards(_lib.i64arr(list(shape)), sum(1 << d for d in dims), DTYPE[dtype], tensors, word_bits, int(asym))


def _without_waiting(x, dims, bits, asym, pack, ticks=0):
    mask = sum(1 << d for d in dims)
    lib, sh = _lib.load(), _lib.i64arr(list(x.shape))
    groups = [1 if d in dims else n for d, n in enumerate(x.shape)]
    s = torch.empty(groups, device=x.device)
    z = torch.empty(groups, device=x.device) if asym else None
    q = torch.empty(*x.shape[:3], x.shape[3] * bits // 32 if pack else x.shape[3], dtype=torch.int32 if pack else torch.int8, device=x.device)
    size = lib.varq_quant_workspace_bytes(sh, mask)
    ws = torch.full(((size + 3) // 4,), -1, dtype=torch.int32, device=x.device)   # (any contents)
    _lib.check(lib.varq_quant_pack_wait(x.data_ptr(), DTYPE[x.dtype], sh, mask, bits, int(asym), 1e-12, q.data_ptr() if pack else None,
                                        None if pack else q.data_ptr(), s.data_ptr(), z.data_ptr() if asym else None, None, ticks, ws.data_ptr(), size,
                                        torch.cuda.current_stream().cuda_stream), 'varq_quant_pack_wait')
    return q, s, z


@pytest.mark.parametrize('shape,dims,dtype', [
    ((2, 4, 16500, 64), (0, 2), torch.bfloat16),      # 828 workgroups of five steps
    ((64, 513, 7, 64), (0, 1), torch.float16),        # two kept indices to a block, the last block half full
    ((3, 11003, 5, 72), (0, 1), torch.float32),       # nine octets of sixteen lanes
    ((1, 4, 70001, 96), (0, 2), torch.bfloat16),      # 18 steps: two beyond the held ones
    ((2, 3, 35001, 128), (0, 2), torch.float32),      # 18 steps of which 8 are held
    ((1, 4, 8300, 256), (0, 2), torch.float16),       # as many groups as a workgroup takes
    ((2, 30, 7000, 64), (0, 2, 3), torch.bfloat16),   # groups of whole rows
    ((32, 30, 421, 64), (0, 1, 3), torch.bfloat16),
])
def test_shared_groups(dev, shape, dims, dtype):
    g = torch.Generator().manual_seed(sum(shape))
    x = (torch.randn(*shape, generator=g) * 2).to(dtype)
    x[..., 3] *= 15
    x[0, 0, 0] = 0
    x[-1, -1, -1] = 40                                # the extreme of its groups, in the last rows of the last workgroup
    for bits, asym, pack in ((8, False, True), (2 if shape[3] % 16 == 0 else 4, True, True), (5, False, False)):
        note('quant shared', shape, dims, dtype, bits, asym, pack)
        assert _shards(x, dims, bits if pack else 8, asym) > 1
        q, s, z = O.quant_reduce(x, dims, bits, asym)
        if pack:
            q = O.pack_last_dim(q, bits)[0]
        for got in (ops.quant_pack(x.to(dev), dims, bits, asym=asym, pack=pack), _without_waiting(x.to(dev), dims, bits, asym, pack)):
            torch.cuda.synchronize()
            assert torch.equal(got[1].cpu(), s)
            assert not asym or torch.equal(got[2].cpu(), z)
            assert torch.equal(got[0].cpu(), q)


def test_shared_groups_in_a_graph(dev):
    """The words that the workgroups exchange are cleared by every replay; K and V of a step in one launch."""
    shape, dims = (64, 129, 16, 64), (0, 1)
    xs = [torch.randn(*shape, device=dev).half() for _ in range(2)]
    assert _shards(xs[0], dims, 8, True, tensors=2) > 1
    ops.quant_pack_pair(*xs, dims, 8, asym=True)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = ops.quant_pack_pair(*xs, dims, 8, asym=True)
    for factor in (4.0, 0.25, 0.5, 2.0):              # (groups that shrink: extremes left by the last replay would show)
        for x in xs:
            x.mul_(factor)
        note('quant shared, replay', factor)
        graph.replay()
        torch.cuda.synchronize()
        for (q, s, z), x in zip(got, xs):
            rq, rs, rz = O.quant_reduce(x.cpu(), dims, 8, True)
            assert torch.equal(s.cpu(), rs) and torch.equal(z.cpu(), rz) and torch.equal(q.cpu(), O.pack_last_dim(rq, 8)[0])


@pytest.mark.parametrize('what', WHAT)
@pytest.mark.parametrize('shape,dims,dtype', [
    ((2, 4, 300, 64), (0, 2), torch.bfloat16),
    ((4, 70, 8, 64), (0, 1), torch.float16),
    ((2, 4, 300, 64), (0, 2), torch.float32),
    ((2, 5, 33, 32), (0, 3), torch.bfloat16),       # groups of whole rows, whose extremes are folded over the columns too
    ((2, 30, 35, 64), (0, 2, 3), torch.float32),
])
def test_infinities_and_nan(dev, shape, dims, dtype, what):
    """The batch behind itself leaves every group what it is and takes workgroups that share it; alone it takes one launch."""
    x = _spoil(torch.randn(*shape, generator=torch.Generator().manual_seed(7)).to(dtype).to(dev), 1 if dims == (0, 1) else 2, what)
    times = (48 << 20) // (x.numel() * x.element_size()) + 1 if 3 in dims else 26000 // math.prod(shape[d] for d in dims) + 1
    for bits, asym in ((8, False), (8, True), (4, True), (2, True)):
        note('quant shared, non-finite', shape, dims, dtype, what, bits, asym)
        q1, s1, z1 = ops.quant_pack(x, dims, bits, asym=asym)
        many = x.repeat(times, 1, 1, 1)
        assert _shards(x, dims, bits, asym) == 1 and _shards(many, dims, bits, asym) > 1
        for q, s, z in (ops.quant_pack(many, dims, bits, asym=asym), _without_waiting(many, dims, bits, asym, True)):
            assert torch.equal(_bits(s1), _bits(s)) and (not asym or torch.equal(_bits(z1), _bits(z)))
            assert torch.equal(q.view(times, *q1.shape), q1.expand(times, *q1.shape))


@pytest.mark.parametrize('shape,dims,dtype,asym', [
    ((2, 3, 35001, 128), (0, 2), torch.float32, False),    # four blocks of 128 and more workgroups
    ((32, 30, 680, 64), (0, 2), torch.bfloat16, True),     # many blocks of a few dozen
    ((32, 30, 680, 64), (0, 2, 3), torch.bfloat16, True),
])
def test_giving_up_on_the_others_reads_the_rows_once_more(dev, shape, dims, dtype, asym):
    """Workgroups that have waited in vain share the others' rows out among themselves.  (When each of them read all rows of its groups, 3 us of
    patience took 5.3 to 28 times the time of waiting; the bar is between that and the 1.1 to 1.25 of one more pass over part of the input.)"""
    x = torch.randn(*shape, generator=torch.Generator().manual_seed(3)).to(dtype).to(dev)

    def median_us(ticks):
        times = []
        for _ in range(15):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            got = _without_waiting(x, dims, 8, asym, True, ticks)
            end.record()
            torch.cuda.synchronize()
            times.append(start.elapsed_time(end) * 1e3)
        return sorted(times)[7], got

    note('quant shared, giving up', shape, dims)
    assert _shards(x, dims, 8, asym) > 1
    (patient, a), (hasty, b) = median_us(1000000), median_us(300)
    assert all(torch.equal(i, j) for i, j in zip(a, b) if i is not None)
    assert hasty < 3 * patient, (patient, hasty)


def _us(f, times=15):
    got = []
    for _ in range(times):
        start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        start.record()
        for _ in range(10):
            f()
        end.record()
        torch.cuda.synchronize()
        got.append(start.elapsed_time(end) * 100)
    return sorted(got)[times // 2]


def test_extremes_of_whole_rows_lie_apart_where_the_workspace_is_small(dev):
    """30 groups whose three launches have 60 chunks leave no room for a line for each extreme; 30 others of as many bytes do.  (Side by side in
    memory the exchange took 1.8 times as long.)"""
    dims = (0, 2, 3)
    x, y = (torch.randn(*shape, device=dev) for shape in ((60, 30, 66, 128), (80, 30, 50, 128)))
    assert _shards(x, dims, 4, True) > 1 and _shards(y, dims, 4, True) > 1
    note('quant shared, room for half a line')
    one, other = _us(lambda: ops.quant_pack(x, dims, 4, asym=True)), _us(lambda: ops.quant_pack(y, dims, 4, asym=True))
    assert one < 1.35 * other, (one, other)
    for t in (x, y):
        s, z = O.quant_reduce(t.cpu(), dims, 4, True)[1:]
        got = ops.quant_pack(t, dims, 4, asym=True)
        assert torch.equal(got[1].cpu(), s) and torch.equal(got[2].cpu(), z)


@pytest.mark.parametrize('shape,dims,dtype,tensors,shared', [
    # heads first, 16 bits, beyond 192 MiB: where the three launches are one round of workgroups, and where they are a little more
    ((39, 8, 6115, 64), (0, 2), torch.float16, 1, False),
    ((526, 16, 64, 128), (0, 2), torch.float16, 2, False),
    ((635, 16, 508, 40), (0, 2, 3), torch.bfloat16, 1, False),
    ((4, 24, 17568, 72), (0, 2), torch.bfloat16, 1, False),      # (of lanes that idle a smaller tensor)
    ((2, 30, 40914, 72), (0, 2), torch.bfloat16, 1, False),      # (of nearly half of them: always)
    ((402, 24, 517, 64), (0, 2), torch.bfloat16, 1, True),
    ((39, 8, 5000, 64), (0, 2), torch.float16, 1, True),
    ((36, 6, 5196, 64), (0, 2), torch.float32, 1, True),
    # few workgroups, 16 bits: up to 24 steps of a workgroup, 16 of them held
    ((4, 3, 12000, 64), (0, 2), torch.float16, 1, True),
    ((284, 3, 680, 128), (0, 2), torch.float16, 1, False),
    ((2, 3, 125467, 128), (0, 2, 3), torch.bfloat16, 1, False),
    ((1, 3, 91810, 128), (0, 2), torch.float32, 1, True),
])
def test_where_the_launches_that_read_twice_are_faster(dev, shape, dims, dtype, tensors, shared):
    """Sizes on either side of the lines, with both ways timed on a device of their own (the figures are at make_shared_plan)."""
    assert (_shards_of(shape, dtype, dims, 4, True, tensors) > 1) == shared


@pytest.mark.parametrize('shape,dims,dtype,tensors,asym,one', [
    ((32, 30, 55, 96), (0, 2), torch.float32, 2, True, True),
    ((8, 476, 30, 96), (0, 1), torch.float32, 1, False, True),
    ((4, 24, 987, 128), (0, 2), torch.float32, 1, False, True),
    ((8, 16, 498, 72), (0, 2), torch.float32, 1, False, True),
    ((16, 16, 494, 72), (0, 2), torch.float32, 1, True, False),
    ((2, 30, 1060, 96), (0, 2), torch.float32, 2, True, False),    # two rounds of workgroups
    ((1, 24, 4270, 128), (0, 2), torch.float16, 1, True, False),
    ((1, 30, 5888, 96), (0, 2), torch.float32, 1, False, False),   # pieces of 32 bytes
])
def test_where_one_workgroup_per_group_is_faster(dev, shape, dims, dtype, tensors, asym, one):
    """Sizes on either side of the line, with both ways timed (the figures are at one_launch_pays)."""
    assert (_shards_of(shape, dtype, dims, 4, asym, tensors) == 1) == one
