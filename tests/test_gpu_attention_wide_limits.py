"""Key limits at sizes where K and V are expanded first: the blocks of 256 queries end at different keys, and a workgroup
takes one each in an order of its own -- pairs that do not fill the eight classes which the workgroups are dealt out to, more
than one window of pairs, limits that rise with the query, fall, or are those of a whole scale schedule.  Held against the kernel that
widens per workgroup (its keys shared out over two) for every output, and against the oracle for some pairs."""
import math

import pytest
import torch

from gpu_util import note
from test_gpu_attention_wide import _check
from var_q_amd import ops, schedules

pytestmark = pytest.mark.gpu


def _limits(order, Lq, Lk, dev):
    if order == 'schedule':
        lim = schedules.kv_limit(list(schedules.INFINITY_PATCH_NUMS[:10]), device=dev)
        assert lim.numel() == Lq == Lk
        return lim
    lim = (torch.arange(Lq, device=dev) * (Lk + 1) // Lq).int()            # 0 .. Lk
    return lim.flip(0).contiguous() if order == 'falling' else lim


@pytest.mark.parametrize('layout', ['BHLc', 'BLHc'])
@pytest.mark.parametrize('D,bits,group,B,H,Lq,Lk,order,dtype', [
    (128, 4, 128, 1, 17, 2521, 2521, 'schedule', 'bf16'),
    (128, 8, 64, 3, 9, 1281, 2048, 'rising', 'bf16'),       # 27 pairs, the last block one query
    (128, 2, 128, 13, 16, 1290, 2050, 'falling', 'bf16'),   # 26 pairs of a class: two windows, of 21 and 5
    (64, 4, 32, 1, 23, 1550, 2111, 'rising', 'fp16'),
    (64, 4, 64, 1, 13, 6150, 2048, 'rising', 'bf16'),
    # few pairs: blocks of 128 queries, the last one full, of one query or of 33 and more; one tile of keys, and two with one key in the second
    (128, 4, 128, 1, 11, 193, 64, 'rising', 'bf16'),
    (128, 2, 64, 2, 5, 256, 65, 'falling', 'bf16'),
    (128, 8, 128, 2, 16, 1441, 1441, 'rising', 'bf16'),
    (64, 4, 32, 1, 16, 680, 680, 'rising', 'fp16'),
    (64, 8, 64, 1, 13, 225, 193, 'falling', 'bf16'),
    (64, 2, 64, 3, 10, 257, 129, 'rising', 'fp16'),
])
def test_blocks_that_end_at_different_keys(dev, D, bits, group, B, H, Lq, Lk, order, dtype, layout):
    dt = torch.float16 if dtype == 'fp16' else torch.bfloat16
    gen = torch.Generator(device=dev).manual_seed(Lq + Lk)
    q = torch.randn(B, H, Lq, D, device=dev, generator=gen).to(dt)
    kq, vq = (ops.quant_pack_rows(torch.randn(B, H, Lk, D, device=dev, generator=gen).bfloat16(), group, bits, True) for _ in range(2))
    lim = _limits(order, Lq, Lk, dev)
    what = 'wide limits %s' % ((D, bits, group, B, H, Lq, Lk, order, dtype, layout),)
    note(what)
    put = (lambda t: t) if layout == 'BHLc' else (lambda t: t.transpose(1, 2).contiguous())
    run = lambda **kw: ops.fused_attn(put(q), *map(put, kq), *map(put, vq), bits, bits, Lk, 1 / math.sqrt(D), kv_limit=lim, layout=layout, **kw)
    out, other = (t if layout == 'BHLc' else t.transpose(1, 2) for t in (run(), run(splits=2)))
    assert bool((out[:, :, lim == 0] == 0).all())
    _check(out, other, q, ops.dequant(*kq, D, bits), ops.dequant(*vq, D, bits), 1 / math.sqrt(D), dt, what, lim)
    assert torch.equal(run(splits=1), put(out))


def test_the_workspace_is_that_of_the_path(dev):
    """Where limits rule the expansion out no memory is taken for it."""
    from var_q_amd import _lib
    lib = _lib.load()
    for B, H, Lq, D in ((2, 16, 4121, 64), (8, 16, 2521, 64)):
        assert lib.varq_fused_attn_expand_bytes(B, H, Lq, Lq, D) > 0 and lib.varq_fused_attn_expand_bytes_limits(B, H, Lq, Lq, D) == 0
    for B, H, Lq, D in ((1, 16, 4121, 64), (8, 16, 6425, 64), (1, 16, 2521, 128)):
        assert lib.varq_fused_attn_expand_bytes_limits(B, H, Lq, Lq, D) >= B * H * Lq * D * 4
