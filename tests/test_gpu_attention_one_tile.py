"""Launches of many (batch, head) pairs with at most 128 queries (the first steps of a schedule at a large batch) run a
kernel with one of each buffer where they have at most 64 keys or more than three pairs to a compute unit; one key more,
or more queries, take the pipelined ones.  The arithmetic is the same, so every pair's output equals bit for bit what the same pair gives in a launch too
small for that rule; two pairs are held against the oracle."""
import math

import pytest
import torch

import varq_oracle as O
from gpu_util import note
from test_gpu_attention import _compare
from var_q_amd import ops

pytestmark = pytest.mark.gpu
H = 17


@pytest.mark.parametrize('Lq,Lk', [(1, 1), (4, 5), (31, 32), (33, 33), (128, 63), (128, 64), (100, 65), (17, 129), (129, 64)])
@pytest.mark.parametrize('B', [19])   # 323 pairs: more than compute units, no multiple of 8
@pytest.mark.parametrize('bits,dtype', [(2, 'fp16'), (4, 'bf16'), (8, 'fp16'), (8, 'bf16')])
@pytest.mark.parametrize('scales', ['g32', 'g64', 'channel'])
def test_small_steps(dev, Lq, Lk, bits, dtype, scales, B):
    D, scale = 64, 0.125
    dt = torch.float16 if dtype == 'fp16' else torch.bfloat16
    gen = torch.Generator(device=dev).manual_seed(Lq * 1000 + Lk)
    q, k, v = (torch.randn(B, H, n, D, device=dev, generator=gen).to(dt) for n in (Lq, Lk, Lk))
    note('one tile', Lq, Lk, bits, dtype, scales)
    lim = (torch.arange(Lq, device=dev, dtype=torch.int32) % (Lk + 1)).contiguous()
    if scales == 'channel':
        # up to three segments with tables of their own
        ends = sorted({(Lk + 2) // 3, (2 * Lk + 2) // 3, Lk})
        cuts = list(zip([0] + ends[:-1], ends))
        def quant(x):
            parts = [ops.quant_pack(x[:, :, a:b].contiguous(), (0, 2), bits, asym=True) for a, b in cuts]
            x = torch.cat([ops.dequant(*p, D, bits) for p in parts], 2)
            return (torch.cat([p[0] for p in parts], 2).contiguous(), *(torch.stack([p[i].reshape(H, D) for p in parts]) for i in (1, 2)), x)
        (kw, ks, kz, kd), (vw, vs, vz, vd) = quant(k), quant(v)
        run = lambda n, **kw_: ops.fused_attn_channel(q[:n], kw[:n], ks, kz, vw[:n], vs, vz, bits, Lk, scale, seg_ends=ends, **kw_)
    else:
        (kw, ks, kz), (vw, vs, vz) = (ops.quant_pack_rows(x, int(scales[1:]), bits, True) for x in (k, v))
        kd, vd = ops.dequant(kw, ks, kz, D, bits), ops.dequant(vw, vs, vz, D, bits)
        run = lambda n, **kw_: ops.fused_attn(q[:n], kw[:n], ks[:n], kz[:n], vw[:n], vs[:n], vz[:n], bits, bits, Lk, scale, **kw_)
    for kw_ in ({}, {'kv_limit': lim}):
        out, few = run(B, **kw_), run(15, **kw_)
        assert torch.equal(out[:15], few)
        live = slice(None) if not kw_ else lim.cpu() > 0
        bias = torch.zeros(Lq, Lk)
        if kw_:
            assert bool((out[:, :, lim == 0] == 0).all())
            bias = bias.masked_fill(torch.arange(Lk)[None] >= lim.cpu()[:, None], -math.inf)
            if not bool(live.any()):
                continue
        for b, h in ((0, 1), (B - 1, H - 1)):
            args = [t[b, h][None, None].cpu() for t in (q, kd, vd)]
            args[0] = args[0][:, :, live]
            ref = O.attention_ref(*args, scale, bias[live], dtype=dt)
            _compare(out[b, h][None, None][:, :, live], ref, O.attention_exact(args[0].float(), *args[1:], scale, bias[live]), 'one tile')


@pytest.mark.parametrize('Lq,Lk', [(1, 65), (33, 127), (64, 128), (128, 191), (65, 257), (5, 700)])
@pytest.mark.parametrize('bits,dtype', [(2, 'fp16'), (4, 'bf16'), (8, 'fp16')])
@pytest.mark.parametrize('scales', ['g32', 'g64', 'channel'])
def test_more_pairs_than_fit_at_once(dev, Lq, Lk, bits, dtype, scales):
    """833 pairs: several tiles through the kernel with one of each buffer (2-bit codes in groups: through two)."""
    test_small_steps(dev, Lq, Lk, bits, dtype, scales, 49)
