"""The memory that K and V take while they are expanded: bounded, with the batch served in parts above the bound; not taken
where the call does not use it; and not missed where the device does not have it."""
import math

import pytest
import torch

from gpu_util import note
from test_gpu_attention_wide import _check
from var_q_amd import PackedKVCache, _lib, ops

pytestmark = pytest.mark.gpu
GIB = 1 << 30


def test_the_size_is_bounded(dev):
    size = _lib.load().varq_fused_attn_expand_bytes
    assert 2 * 16 * 10521 * 512 <= size(2, 16, 4096, 10521, 128) < 2 * 16 * 10560 * 512 + 70e6       # all at once
    for B, H, Lq, Lk, D in ((16, 24, 4096, 10521, 128), (64, 30, 1600, 4121, 64), (1000, 8, 1300, 2048, 128)):
        assert GIB // 2 < size(B, H, Lq, Lk, D) <= GIB + (70 << 20)
    assert size(2, 64, 4096, 40000, 128) == 0                                                         # not one batch entry


@pytest.mark.parametrize('layout', ['BHLc', 'BLHc'])
def test_token_scales_in_parts(dev, layout):
    B, H, Lq, Lk, D = 9, 24, 1285, 10500, 128            # 129 MB a batch entry: parts of 5 and 4
    note('expanded in parts: token scales', layout)
    gen = torch.Generator(device=dev).manual_seed(1)
    q = torch.randn(B, H, Lq, D, device=dev, generator=gen).bfloat16()
    kq, vq = (ops.quant_pack_rows(torch.randn(B, H, Lk, D, device=dev, generator=gen).bfloat16(), 128, 4, True) for _ in range(2))
    put = (lambda t: t) if layout == 'BHLc' else (lambda t: t.transpose(1, 2).contiguous())
    run = lambda **kw: put(ops.fused_attn(put(q), *map(put, kq), *map(put, vq), 4, 4, Lk, 1 / math.sqrt(D), layout=layout, **kw))
    kd, vd = ({b: ops.dequant(*(t[b:b + 1] for t in x), D, 4)[0] for b in (0, 4, 5, 8)} for x in (kq, vq))
    _check(run(), run(splits=2), q, _Some(kd), _Some(vd), 1 / math.sqrt(D), torch.bfloat16, 'parts', pairs=((0, 0), (4, 23), (5, 0), (8, 23)))


class _Some:
    """The batch entries that are compared with the oracle."""

    def __init__(self, entries):
        self.entries = entries

    def __getitem__(self, at):
        return self.entries[at[0]][at[1]]


def test_tables_in_parts(dev):
    B, H, Lq, steps, D = 18, 24, 1540, [2000, 8500], 64
    Lk = sum(steps)
    note('expanded in parts: tables')
    gen = torch.Generator(device=dev).manual_seed(2)
    q = torch.randn(B, H, Lq, D, device=dev, generator=gen).half()
    packed = []
    for _ in range(2):
        parts = [ops.quant_pack(torch.randn(B, H, n, D, device=dev, generator=gen).half() * (1 + i), (0, 2), 8, True) for i, n in enumerate(steps)]
        table = lambda i: torch.stack([p[i].reshape(H, D) for p in parts]).contiguous()
        packed.append((torch.cat([p[0] for p in parts], 2).contiguous(), table(1), table(2)))
    hm = torch.randperm(H, generator=torch.Generator().manual_seed(1)).int().to(dev)
    run = lambda **kw: ops.fused_attn_channel(q, *packed[0], *packed[1], 8, Lk, 0.125, seg_ends=[steps[0], Lk], head_map=hm, **kw)
    out, other = run(), run(splits=2)
    assert not bool(torch.isnan(out).any()) and float((out.float() - other.float()).abs().max()) <= 1e-2 * max(1.0, float(other.abs().max()))


def test_bit_width_classes_in_parts(dev):
    B, H, Lq, Lk, D = 9, 24, 1285, 10500, 128
    note('expanded in parts: classes')
    gen = torch.Generator(device=dev).manual_seed(3)
    cache = PackedKVCache(B, H, Lk, D, [2, 8, 4, 8, 2, 4] * 4, 64, dev)
    cache.append(*(torch.randn(B, H, Lk, D, device=dev, generator=gen).bfloat16() for _ in range(2)))
    q = torch.randn(B, H, Lq, D, device=dev, generator=gen).bfloat16()
    out = cache.attend(q, 0.09)
    cache.splits = 2
    other = cache.attend(q, 0.09)
    assert not bool(torch.isnan(out).any()) and float((out.float() - other.float()).abs().max()) <= 1e-2 * max(1.0, float(other.abs().max()))


def _call(dev, seed=4):
    B, H, Lq, Lk, D = 2, 16, 1600, 10000, 128
    gen = torch.Generator(device=dev).manual_seed(seed)
    q = torch.randn(B, H, Lq, D, device=dev, generator=gen).bfloat16()
    kq, vq = (ops.quant_pack_rows(torch.randn(B, H, Lk, D, device=dev, generator=gen).bfloat16(), 128, 4, True) for _ in range(2))
    return lambda **kw: ops.fused_attn(q, *kq, *vq, 4, 4, Lk, 1 / math.sqrt(D), **kw)


def _peak(f):
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    out = f()
    torch.cuda.synchronize()
    return out, torch.cuda.max_memory_allocated() - before


def test_exact_codes_take_no_memory_for_it(dev):
    note('expanded: exact codes')
    run = _call(dev)
    assert _peak(run)[1] > 160e6 and _peak(lambda: run(exact_codes=True))[1] < 120e6 and _peak(lambda: run(splits=2))[1] < 120e6


def test_a_device_without_room_for_it(dev):
    """The allocator is held to what there is and 100 MB: the 173 MB of the expanded K and V are refused, and the call is
    served as it was with the smaller workspace."""
    note('expanded: no room')
    run = _call(dev)
    want = run()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(dev).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + 100e6) / total, dev)
    try:
        out, peak = _peak(run)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0, dev)
    assert peak < 110e6
    assert float((out.float() - want.float()).abs().max()) <= 1e-2 * max(1.0, float(want.abs().max()))
    assert torch.equal(run(), want)
