"""The kernel for few queries at the forms it takes: both head dims, one and two scale groups per key, K and V grouped
differently, all bit-widths, fp16, one and two columns of queries and several tiles of them, four and eight wavefronts, ends of
blocks and of the cache, zero-points outside what it holds in fp16, both layouts, spare rows, key limits -- against the oracle
(the bar of test_gpu_attention.py) and against the kernel for many queries on the same inputs (`splits=1`): the operands are the same
roundings, so the two differ by the order of their sums and by the 16-bit rounding of their weights."""
import math

import pytest
import torch

import varq_oracle as O
from gpu_util import note
from test_gpu_attention import _compare, _exact_fp64
from var_q_amd import _lib, ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('Lq,Lk', [(1, 1), (3, 31), (16, 32), (17, 65), (5, 129), (16, 257), (33, 300), (16, 600), (128, 129), (70, 500), (2, 1025), (20, 2100)])
@pytest.mark.parametrize('D,gk,gv,dtype', [(128, 128, 128, 'bf16'), (128, 64, 64, 'bf16'), (64, 64, 64, 'fp16'), (64, 32, 64, 'bf16'), (64, 32, 32, 'fp16')])
@pytest.mark.parametrize('bits', [4, 2, 8])
def test_forms(dev, bits, D, gk, gv, dtype, Lq, Lk):
    seed = bits + D + gk + Lq * 7 + Lk
    gen = torch.Generator().manual_seed(seed)
    dt = torch.float16 if dtype == 'fp16' else torch.bfloat16
    B, H, scale = 2, 3, 1 / math.sqrt(D)
    layout, limit, spare = ('BHLc', 'BLHc')[seed % 2], seed % 3 == 0, 9 * (seed % 5 == 0)
    far = seed % 4 == 0   # (the values of such zero-points have to fit fp16: no heavy tails there)
    k, v = (O.synth_kv((B, H, Lk, D), seed + i, 'normal' if far else 'student4').to(dt) for i in (1, 2))
    q = torch.randn(B, H, Lq, D, generator=gen).to(dt)
    kq, ks, kz = O.quant_groupwise(k, gk, bits, True)
    vq, vs, vz = O.quant_groupwise(v, gv, bits, True)
    kz, vz = kz.clone(), vz.clone()
    if far:      # beyond what fp16 counts, and fractions, in some keys of some groups
        kz[:, 1, Lk // 2:, -1:], vz[:, 2, :Lk // 3 + 1, :1] = 1500.0, -1200.0
        kz[:, 0, -1:] += 0.25
        vz[:, 0, Lk // 2:Lk // 2 + 3, -1:] -= 0.5
    kd, vd = O.dequant_groupwise(kq, ks, kz, gk), O.dequant_groupwise(vq, vs, vz, gv)
    lim = bias = None
    if limit:
        lim = torch.randint(1, Lk + 1, (Lq,), generator=gen).int()
        bias = torch.zeros(Lq, Lk).masked_fill(torch.arange(Lk)[None] >= lim[:, None], -math.inf)
    rows = [O.pack_last_dim(kq, bits)[0], ks, kz, O.pack_last_dim(vq, bits)[0], vs, vz]
    if spare:
        rows = [torch.cat([t, torch.full((B, H, spare, t.shape[3]), 0x7f if t.dtype == torch.int32 else 1e30, dtype=t.dtype)], 2) for t in rows]
    turn = (lambda t: t.transpose(1, 2).contiguous()) if layout == 'BLHc' else (lambda t: t.contiguous())
    rows = [turn(t).to(dev) for t in rows]
    assert _lib.load().varq_fused_attn_key_shares(B, H, Lq, Lk, D, gk, gv) >= 1
    note('few queries, forms', bits, D, gk, gv, dtype, Lq, Lk, layout, limit, spare)
    run = lambda n: ops.fused_attn(turn(q).to(dev), *rows, bits, bits, Lk, scale, kv_limit=None if lim is None else lim.to(dev), splits=n, layout=layout)
    few, many = run(0), run(1)
    torch.cuda.synchronize()
    if layout == 'BLHc':
        few, many = few.transpose(1, 2), many.transpose(1, 2)
    _compare(few, O.attention_ref(q, kd, vd, scale, bias, dtype=dt), _exact_fp64(q, kd, vd, scale, bias, dev), 'few queries, forms')
    # two roundings of the result and, on both sides, weights rounded to 2^-9 (2^-12) of themselves: within four steps of the largest
    span = max(1.0, float(many.float().abs().max()))
    assert float((few.float() - many.float()).abs().max()) <= span * (2 ** -9 if dtype == 'fp16' else 2 ** -6)


@pytest.mark.parametrize('Lq', [16, 40])
def test_scales_that_are_not_finite(dev, Lq):
    """A NaN or an infinity in one group of one key is one in every channel (K) or in the group's channels (V) of that (batch, head) alone."""
    B, H, Lk, D, group = 2, 3, 700, 128, 64
    gen = torch.Generator(device=dev).manual_seed(3)
    q = torch.randn(B, H, Lq, D, device=dev, generator=gen).bfloat16()
    kq, vq = ([t.clone() for t in ops.quant_pack_rows(torch.randn(B, H, Lk, D, device=dev, generator=gen).bfloat16(), group, 4, True)] for _ in range(2))
    note('few queries, scales not finite', Lq)
    kq[1][0, 1, 650, 1] = math.nan
    kq[1][1, 2, 0, 0] = math.inf
    vq[1][1, 0, 333, 1] = math.nan
    out = torch.isfinite(ops.fused_attn(q, *kq, *vq, 4, 4, Lk, 0.09))
    want = torch.ones_like(out)
    want[0, 1] = want[1, 2] = want[1, 0, :, 64:] = False
    assert torch.equal(out, want)
