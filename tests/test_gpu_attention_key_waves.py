"""Launches that leave compute units idle: two or four wavefronts of a workgroup share the keys of its queries.  At the edges of
the blocks of 128 and 64 queries, of the tiles of 64 and 128 keys and of the 32 keys of a wavefront (shares without any key among
them), held against the same kernel with the keys shared out over two workgroups and against the oracle."""
import math

import pytest
import torch

from gpu_util import note
from test_gpu_attention_wide import _check
from var_q_amd import PackedKVCache, _lib, ops

pytestmark = pytest.mark.gpu

EDGES = [(129, 65), (192, 96), (193, 97), (256, 128), (257, 129), (130, 161), (300, 193), (400, 1025)]


def _waves(B, H, Lq, Lk, D, limits):
    return _lib.load().varq_fused_attn_key_waves(B, H, Lq, Lk, D, limits)


def _inputs(dev, B, H, Lq, Lk, D, dt):
    gen = torch.Generator(device=dev).manual_seed(Lq + Lk + D)
    k, v = (torch.randn(B, H, Lk, D, device=dev, generator=gen) for _ in range(2))
    k[..., 3] *= 15.0
    return torch.randn(B, H, Lq, D, device=dev, generator=gen).to(dt), k.to(dt), v.to(dt)


@pytest.mark.parametrize('Lq,Lk', EDGES)
@pytest.mark.parametrize('D,bits,group,B,H,dtype,waves', [
    (128, 4, 128, 1, 6, 'bf16', 4), (128, 8, 64, 3, 13, 'bf16', 2), (128, 2, 32, 1, 11, 'bf16', 4),
    (64, 4, 32, 2, 7, 'fp16', 4), (64, 8, 64, 3, 13, 'bf16', 2), (64, 2, 64, 1, 9, 'fp16', 4),
])
def test_token_scales(dev, D, bits, group, B, H, dtype, waves, Lq, Lk):
    dt = torch.float16 if dtype == 'fp16' else torch.bfloat16
    q, k, v = _inputs(dev, B, H, Lq, Lk, D, dt)
    kq, vq = (ops.quant_pack_rows(t, group, bits, True) for t in (k, v))
    kd, vd = (ops.dequant(*t, D, bits) for t in (kq, vq))
    what = 'key waves %s' % ((D, bits, group, B, H, Lq, Lk, dtype),)
    rising = torch.clamp((torch.arange(Lq, device=dev) + 1) * Lk // Lq, max=Lk).int().contiguous()
    taken = set()
    for layout in ('BHLc', 'BLHc'):
        put = (lambda t: t) if layout == 'BHLc' else (lambda t: t.transpose(1, 2).contiguous())
        run = lambda **kw: put(ops.fused_attn(put(q), *map(put, kq), *map(put, vq), bits, bits, Lk, 1 / math.sqrt(D), layout=layout, **kw))
        for lim in (None, rising):
            note(what, layout, lim is not None)
            taken.add(_waves(B, H, Lq, Lk, D, lim is not None))
            _check(run(kv_limit=lim), run(kv_limit=lim, splits=2), q, kd, vd, 1 / math.sqrt(D), dt, what, lim)
    assert taken & {2, 4}


def test_both_numbers_are_reached():
    for D in (64, 128):
        for limits in (0, 1):
            assert {2, 4} <= {_waves(B, 12, Lq, Lk, D, limits) for B in (1, 3, 6) for Lq, Lk in EDGES}


@pytest.mark.parametrize('Lq,Lk', EDGES)
@pytest.mark.parametrize('D,bits,asym', [(128, 8, False), (128, 4, True), (64, 8, False), (64, 2, True)])
def test_tables(dev, D, bits, asym, Lq, Lk):
    B, H = 1, 7
    dt = torch.float16 if D == 64 else torch.bfloat16
    q, k, v = _inputs(dev, B, H, Lq, Lk, D, dt)
    ends = sorted({1, 5, Lk // 3, Lk // 2 + 7, Lk})
    cuts = list(zip([0] + ends[:-1], ends))
    def quant(x):
        parts = [ops.quant_pack(x[:, :, a:b].contiguous(), (0, 2), bits, asym=asym) for a, b in cuts]
        table = lambda i: torch.stack([p[i].reshape(H, D) for p in parts])
        return (torch.cat([p[0] for p in parts], 2).contiguous(), table(1), table(2) if asym else None), torch.cat([ops.dequant(*p, D, bits) for p in parts], 2)
    (kq, kd), (vq, vd) = quant(k), quant(v)
    what = 'key waves, tables %s' % ((D, bits, asym, Lq, Lk),)
    note(what)
    assert _waves(B, H, Lq, Lk, D, 0) > 1
    run = lambda **kw: ops.fused_attn_channel(q, *kq, *vq, bits, Lk, 1 / math.sqrt(D), seg_ends=ends, **kw)
    _check(run(), run(splits=2), q, kd, vd, 1 / math.sqrt(D), dt, what)


@pytest.mark.parametrize('D,group', [(128, 64), (64, 32)])
@pytest.mark.parametrize('B', [1, 7])
def test_several_bit_widths(dev, D, group, B):
    H, Lq, Lk, bits = 6, 200, 333, [2, 8, 4, 4, 8, 2]
    q, k, v = _inputs(dev, B, H, Lq, Lk, D, torch.bfloat16)
    cache = PackedKVCache(B, H, Lk, D, bits, group, dev)
    cache.append(k, v)
    note('key waves, several bit-widths', D, B)
    assert _waves(B, H, Lq, Lk, D, 0) > 1
    out = cache.attend(q, 1 / math.sqrt(D))
    for h, b in enumerate(bits):
        one = lambda t: t[:, h:h + 1].contiguous()
        kq, vq = (ops.quant_pack_rows(one(t), group, b, True) for t in (k, v))
        want = ops.fused_attn(one(q), *kq, *vq, b, b, Lk, 1 / math.sqrt(D), splits=2)
        _check(one(out), want, one(q), ops.dequant(*kq, D, b), ops.dequant(*vq, D, b), 1 / math.sqrt(D), torch.bfloat16, (h, b), pairs=((0, 0),))


@pytest.mark.parametrize('at', [0, 40, 100, 199])
def test_a_nan_in_one_share(dev, at):
    D, B, H, Lq, Lk = 128, 1, 8, 150, 200
    q, k, v = _inputs(dev, B, H, Lq, Lk, D, torch.bfloat16)
    (kw, ks, kz), vq = ops.quant_pack_rows(k, 128, 8, True), ops.quant_pack_rows(v, 128, 8, True)
    ks[0, 3, at] = math.nan
    note('key waves, NaN', at)
    assert _waves(B, H, Lq, Lk, D, 0) > 1
    out = ops.fused_attn(q, kw, ks, kz, *vq, 8, 8, Lk, 1 / math.sqrt(D))
    bad = torch.isnan(out).all(-1)
    assert bool(bad[0, 3].all()) and not bool(torch.isnan(out[0, [0, 1, 2, 4, 5, 6, 7]]).any())
