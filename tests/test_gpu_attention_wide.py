"""Attention of many queries over a packed cache that is expanded to matrix operands once
(wide_attn.hip): the shapes below are above the line from which the library takes it, at the
edges of its tiles (64 keys, 256 queries, 32 queries of a wavefront) and of its rounds over the
compute units.  Every output is held against the kernel that widens per workgroup (`splits=2`: shares of the keys are its
alone) and against this path without blocks shared out (`splits=1`), two (batch, head) pairs of each against the oracle."""
import math

import pytest
import torch

import varq_oracle as O
from gpu_util import note
from test_gpu_attention import _compare
from var_q_amd import ops
from var_q_amd._lib import VarqError

pytestmark = pytest.mark.gpu


def _check(out, one, q, kd, vd, scale, dtype, what, limit=None, pairs=((0, 0), (-1, -1))):
    span = max(1.0, float(one.abs().max()))
    assert not bool(torch.isnan(out).any())
    assert float((out.double() - one.double()).abs().max()) <= 1e-2 * span, what
    for b, h in pairs:
        bias = None
        if limit is not None:
            bias = torch.zeros(q.shape[2], kd.shape[2]).masked_fill(torch.arange(kd.shape[2])[None] >= limit.cpu()[:, None], -math.inf)
        args = (q[b, h][None, None].cpu(), kd[b, h][None, None].cpu(), vd[b, h][None, None].cpu(), scale, bias)
        ref = O.attention_ref(*args, dtype=dtype)
        live = slice(None) if limit is None else limit.cpu() > 0
        _compare(out[b, h][None, None][:, :, live], ref[:, :, live], O.attention_exact(args[0].float(), *args[1:])[:, :, live], what)


@pytest.mark.parametrize('D,bits,group,B,H,Lq,Lk,dtype', [
    (128, 4, 128, 2, 14, 1281, 2048, 'bf16'),    # 168 blocks, the last of each head one query; whole tiles
    (128, 8, 64, 2, 16, 1537, 2049, 'bf16'),     # one key in the last tile
    (128, 2, 32, 1, 27, 1536, 2111, 'bf16'),     # 63 keys in the last tile
    (128, 4, 64, 4, 13, 1290, 2200, 'bf16'),     # one whole round and 56 blocks shared out
    (64, 4, 32, 2, 17, 1550, 2100, 'fp16'),
    (64, 8, 64, 3, 9, 1600, 2300, 'bf16'),
    (64, 2, 64, 1, 33, 1792, 2080, 'fp16'),
])
def test_token_scales(dev, D, bits, group, B, H, Lq, Lk, dtype):
    dt = torch.float16 if dtype == 'fp16' else torch.bfloat16
    gen = torch.Generator(device=dev).manual_seed(Lq + Lk)
    x = torch.randn(2, B, H, Lk, D, device=dev, generator=gen)
    x[..., 3] *= 15.0
    q = torch.randn(B, H, Lq, D, device=dev, generator=gen).to(dt)
    kq, vq = (ops.quant_pack_rows(t.bfloat16().contiguous(), group, bits, True) for t in x)
    kd, vd = (ops.dequant(*t, D, bits) for t in (kq, vq))
    what = 'wide %s' % ((D, bits, group, B, H, Lq, Lk, dtype),)
    note(what)
    run = lambda **kw: ops.fused_attn(q, *kq, *vq, bits, bits, Lk, 1 / math.sqrt(D), **kw)
    out = run()
    _check(out, run(splits=2), q, kd, vd, 1 / math.sqrt(D), dt, what)
    _check(run(splits=1), out, q, kd, vd, 1 / math.sqrt(D), dt, what)
    # the same with key limits (none, one, tile edges, all) and with the output tokens-first
    limit = torch.tensor([Lk, 0, 1, 64, 65, 33, Lk - 1, 2047], dtype=torch.int32, device=dev)[torch.arange(Lq, device=dev) // 50 % 8].contiguous()
    note(what, 'limits')
    out = run(kv_limit=limit, out_layout='BLHc').transpose(1, 2)
    assert bool((out[:, :, limit == 0] == 0).all())
    _check(out, run(kv_limit=limit, splits=2), q, kd, vd, 1 / math.sqrt(D), dt, what + ' limits', limit)
    # tokens-first cache and queries: the same bits
    t = lambda z: z.transpose(1, 2).contiguous()
    note(what, 'tokens first')
    again = ops.fused_attn(t(q), *(t(z) for z in kq), *(t(z) for z in vq), bits, bits, Lk, 1 / math.sqrt(D), layout='BLHc')
    assert torch.equal(again.transpose(1, 2), run())


@pytest.mark.parametrize('D,bits,asym,dtype', [(128, 8, False, 'bf16'), (128, 4, True, 'bf16'), (64, 2, True, 'fp16'), (64, 8, False, 'bf16')])
def test_stepwise_tables_and_head_map(dev, D, bits, asym, dtype):
    """A table per step, boundaries inside tiles; packed heads in another order than the query heads."""
    dt = torch.float16 if dtype == 'fp16' else torch.bfloat16
    B, H, Lq, steps = 2, 15, 1600, [1, 4, 60, 300, 1000, 735]
    Lk = sum(steps)
    gen = torch.Generator(device=dev).manual_seed(D + bits)
    q = torch.randn(B, H, Lq, D, device=dev, generator=gen).to(dt)
    packed, deq = [], []
    for _ in range(2):
        parts = [ops.quant_pack(torch.randn(B, H, n, D, device=dev, generator=gen).bfloat16() * (1 + i), (0, 2), bits, asym) for i, n in enumerate(steps)]
        table = lambda i: None if parts[0][i] is None else torch.stack([p[i].reshape(H, D) for p in parts]).contiguous()
        packed.append((torch.cat([p[0] for p in parts], 2).contiguous(), table(1), table(2)))
        deq.append(torch.cat([ops.dequant(*p, D, bits) for p in parts], 2))
    perm = torch.randperm(H, generator=torch.Generator().manual_seed(1))
    ends = [sum(steps[:i + 1]) for i in range(len(steps))]
    what = 'wide tables %s' % ((D, bits, asym, dtype),)
    note(what)
    run = lambda **kw: ops.fused_attn_channel(q, *packed[0], *packed[1], bits, Lk, 0.05, seg_ends=ends,
                                              head_map=perm.int().to(dev), **kw)
    back = torch.empty_like(perm)
    back[perm] = torch.arange(H)
    _check(run(splits=1), run(splits=2), q, deq[0][:, back.to(dev)], deq[1][:, back.to(dev)], 0.05, dt, what)
    _check(run(), run(splits=2), q, deq[0][:, back.to(dev)], deq[1][:, back.to(dev)], 0.05, dt, what)


@pytest.mark.parametrize('D,k_group,v_group', [(128, 16, 16), (128, 4, 4), (128, 64, 32), (128, 128, 64), (64, 8, 8), (64, 16, 32)])
def test_groups_without_a_kernel_are_refused_at_every_size(dev, D, k_group, v_group):
    """... also where the call is large enough for the path that could widen some of them."""
    B, H, Lq, Lk = 2, 16, 1600, 2100
    q = torch.zeros(B, H, Lq, D, dtype=torch.bfloat16, device=dev)
    words, scale = torch.zeros(B, H, Lk, D // 8, dtype=torch.int32, device=dev), lambda g: torch.ones(B, H, Lk, D // g, device=dev)
    for splits in (0, 1):
        note('wide: groups', D, k_group, v_group, splits)
        with pytest.raises(VarqError):
            ops.fused_attn(q, words, scale(k_group), None, words, scale(v_group), None, 4, 4, Lk, 0.1, splits=splits)


def test_logits_that_climb_move_the_reference(dev):
    """The softmax reference is set from the first keys; later logits far above it redo their block."""
    B, H, Lq, Lk, D = 2, 14, 1300, 2100, 128
    gen = torch.Generator(device=dev).manual_seed(9)
    k = torch.randn(B, H, Lk, D, device=dev, generator=gen) * torch.linspace(0.1, 6.0, Lk, device=dev)[:, None]
    v = torch.randn(B, H, Lk, D, device=dev, generator=gen)
    q = torch.randn(B, H, Lq, D, device=dev, generator=gen).bfloat16()
    kq, vq = (ops.quant_pack_rows(t.bfloat16(), 128, 8, True) for t in (k, v))
    note('wide climbing logits')
    run = lambda **kw: ops.fused_attn(q, *kq, *vq, 8, 8, Lk, 1.0, **kw)
    _check(run(), run(splits=2), q, ops.dequant(*kq, D, 8), ops.dequant(*vq, D, 8), 1.0, torch.bfloat16, 'wide climbing logits')
