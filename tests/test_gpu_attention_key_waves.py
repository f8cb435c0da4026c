"""Launches that leave compute units idle: two or four wavefronts of a workgroup share the keys of its queries.  At the edges of
the blocks of 128 and 64 queries, of the tiles of 64 and 128 keys and of the 32 keys of a wavefront (shares without any key among
them), held against the same kernel with the keys shared out over two workgroups and against the oracle.  Every case has so many pairs that the
library takes the number of wavefronts that it names."""
import math

import pytest
import torch

from gpu_util import note
from test_gpu_attention_wide import _check
from var_q_amd import PackedKVCache, _lib, ops

pytestmark = pytest.mark.gpu

EDGES = [(129, 65), (192, 96), (193, 97), (256, 128), (257, 129), (130, 161), (300, 193), (400, 1025)]
LIMIT_EDGES = [(193, 193), (256, 256), (257, 257), (385, 385), (449, 449), (400, 1025)]


def _waves(B, H, Lq, Lk, D, limits, nseg=1):
    return _lib.load().varq_fused_attn_key_waves(B, H, Lq, Lk, D, nseg, limits)


def _pairs(waves, Lq, Lk, D, limits=0, nseg=1):
    """The fewest pairs (five at least) whose keys that many wavefronts share."""
    found = [n for n in range(5, 129) if _waves(1, n, Lq, Lk, D, limits, nseg) == waves]
    assert found, (waves, Lq, Lk, D, limits, nseg)
    return found[0]


def _inputs(dev, B, H, Lq, Lk, D, dt):
    gen = torch.Generator(device=dev).manual_seed(Lq + Lk + D)
    k, v = (torch.randn(B, H, Lk, D, device=dev, generator=gen) for _ in range(2))
    k[..., 3] *= 15.0
    return torch.randn(B, H, Lq, D, device=dev, generator=gen).to(dt), k.to(dt), v.to(dt)


def _rising(Lq, Lk, dev):
    return torch.clamp((torch.arange(Lq, device=dev) + 1) * Lk // Lq, max=Lk).int().contiguous()


FORMS = [(128, 4, 128, 'bf16'), (128, 8, 64, 'bf16'), (128, 2, 32, 'bf16'), (64, 4, 32, 'fp16'), (64, 8, 64, 'bf16'), (64, 2, 64, 'fp16')]


def _token_scales(dev, D, bits, group, dtype, waves, Lq, Lk, limits):
    dt = torch.float16 if dtype == 'fp16' else torch.bfloat16
    H = _pairs(waves, Lq, Lk, D, limits)
    B, H = (2, H // 2) if H % 2 == 0 else (1, H)
    assert _waves(B, H, Lq, Lk, D, limits) == waves
    q, k, v = _inputs(dev, B, H, Lq, Lk, D, dt)
    kq, vq = (ops.quant_pack_rows(t, group, bits, True) for t in (k, v))
    kd, vd = (ops.dequant(*t, D, bits) for t in (kq, vq))
    what = 'key waves %s' % ((D, bits, group, B, H, Lq, Lk, dtype, waves, limits),)
    lim = _rising(Lq, Lk, dev) if limits else None
    for layout in ('BHLc', 'BLHc'):
        put = (lambda t: t) if layout == 'BHLc' else (lambda t: t.transpose(1, 2).contiguous())
        run = lambda **kw: put(ops.fused_attn(put(q), *map(put, kq), *map(put, vq), bits, bits, Lk, 1 / math.sqrt(D), layout=layout, kv_limit=lim, **kw))
        note(what, layout)
        _check(run(), run(splits=2), q, kd, vd, 1 / math.sqrt(D), dt, what, lim)


@pytest.mark.parametrize('waves', [2, 4])
@pytest.mark.parametrize('Lq,Lk', EDGES)
@pytest.mark.parametrize('D,bits,group,dtype', FORMS)
def test_token_scales(dev, D, bits, group, dtype, Lq, Lk, waves):
    _token_scales(dev, D, bits, group, dtype, waves, Lq, Lk, 0)


@pytest.mark.parametrize('waves', [2, 4])
@pytest.mark.parametrize('Lq,Lk', LIMIT_EDGES)
@pytest.mark.parametrize('D,bits,group,dtype', FORMS)
def test_token_scales_under_limits(dev, D, bits, group, dtype, Lq, Lk, waves):
    _token_scales(dev, D, bits, group, dtype, waves, Lq, Lk, 1)


@pytest.mark.parametrize('Lq,Lk', EDGES)
@pytest.mark.parametrize('D,bits,group,dtype', FORMS)
def test_few_pairs_under_limits(dev, D, bits, group, dtype, Lq, Lk):
    """Up to 128 keys none are shared under limits, beyond them by four wavefronts where there are few pairs."""
    _token_scales(dev, D, bits, group, dtype, 1 if Lk <= 128 else 4, Lq, Lk, 1)


@pytest.mark.parametrize('waves', [2, 4])
@pytest.mark.parametrize('Lq,Lk,limits', [e + (0,) for e in EDGES] + [(257, 257, 1), (449, 449, 1)])
@pytest.mark.parametrize('D,bits,asym', [(128, 8, False), (128, 4, True), (64, 8, False), (64, 2, True)])
def test_tables(dev, D, bits, asym, Lq, Lk, limits, waves):
    ends = sorted({1, 5, Lk // 3, Lk // 2 + 7, Lk})
    B, H = 1, _pairs(waves, Lq, Lk, D, limits, len(ends))
    dt = torch.float16 if D == 64 else torch.bfloat16
    q, k, v = _inputs(dev, B, H, Lq, Lk, D, dt)
    cuts = list(zip([0] + ends[:-1], ends))
    def quant(x):
        parts = [ops.quant_pack(x[:, :, a:b].contiguous(), (0, 2), bits, asym=asym) for a, b in cuts]
        table = lambda i: torch.stack([p[i].reshape(H, D) for p in parts])
        return (torch.cat([p[0] for p in parts], 2).contiguous(), table(1), table(2) if asym else None), torch.cat([ops.dequant(*p, D, bits) for p in parts], 2)
    (kq, kd), (vq, vd) = quant(k), quant(v)
    what = 'key waves, tables %s' % ((D, bits, asym, Lq, Lk, limits, waves),)
    note(what)
    lim = _rising(Lq, Lk, dev) if limits else None
    run = lambda **kw: ops.fused_attn_channel(q, *kq, *vq, bits, Lk, 1 / math.sqrt(D), seg_ends=ends, kv_limit=lim, **kw)
    _check(run(), run(splits=2), q, kd, vd, 1 / math.sqrt(D), dt, what, lim)


@pytest.mark.parametrize('waves', [2, 4])
@pytest.mark.parametrize('Lq,Lk,limits', [(200, 333, 0), (257, 129, 0), (257, 257, 1), (449, 449, 1)])
@pytest.mark.parametrize('D,group,dt', [(128, 64, torch.bfloat16), (64, 32, torch.bfloat16), (64, 64, torch.float16)])
def test_several_bit_widths(dev, D, group, dt, Lq, Lk, limits, waves):
    B, H = 1, _pairs(waves, Lq, Lk, D, limits)
    bits = [(2, 8, 4, 4, 8)[h % 5] for h in range(H)]
    q, k, v = _inputs(dev, B, H, Lq, Lk, D, dt)
    cache = PackedKVCache(B, H, Lk, D, bits, group, dev)
    cache.append(k, v)
    note('key waves, several bit-widths', D, group, dt, Lq, Lk, limits, waves)
    lim = _rising(Lq, Lk, dev) if limits else None
    out = cache.attend(q, 1 / math.sqrt(D), kv_limit=lim)
    for h in (0, 1, 2, H - 2, H - 1):
        one = lambda t: t[:, h:h + 1].contiguous()
        kq, vq = (ops.quant_pack_rows(one(t), group, bits[h], True) for t in (k, v))
        want = ops.fused_attn(one(q), *kq, *vq, bits[h], bits[h], Lk, 1 / math.sqrt(D), splits=2, kv_limit=lim)
        _check(one(out), want, one(q), ops.dequant(*kq, D, bits[h]), ops.dequant(*vq, D, bits[h]), 1 / math.sqrt(D), dt, (h, bits[h]), lim, pairs=((0, 0),))


@pytest.mark.parametrize('waves', [2, 4])
@pytest.mark.parametrize('at', [0, 40, 100, 199])
def test_a_nan_in_one_share(dev, at, waves):
    D, B, Lq, Lk = 128, 1, 150, 200
    H = _pairs(waves, Lq, Lk, D)
    q, k, v = _inputs(dev, B, H, Lq, Lk, D, torch.bfloat16)
    (kw, ks, kz), vq = ops.quant_pack_rows(k, 128, 8, True), ops.quant_pack_rows(v, 128, 8, True)
    ks[0, 3, at] = math.nan
    note('key waves, NaN', at, waves)
    out = ops.fused_attn(q, kw, ks, kz, *vq, 8, 8, Lk, 1 / math.sqrt(D))
    bad = torch.isnan(out).all(-1)
    assert bool(bad[0, 3].all()) and not bool(torch.isnan(out[0, [h for h in range(H) if h != 3]]).any())


@pytest.mark.parametrize('waves', [2, 4])
@pytest.mark.parametrize('D,bits,group,dtype', [(128, 4, 128, 'bf16'), (64, 8, 64, 'fp16')])
@pytest.mark.parametrize('bad', [math.nan, math.inf])
def test_a_nan_behind_the_limit_in_another_share(dev, D, bits, group, dtype, bad, waves):
    """Queries that see the first share's keys alone, among others that see all: what the other shares hold of V is not theirs."""
    dt = torch.float16 if dtype == 'fp16' else torch.bfloat16
    Lq = Lk = 449
    B, H = 1, _pairs(waves, Lq, Lk, D, 1)
    q, k, v = _inputs(dev, B, H, Lq, Lk, D, dt)
    kq, (vw, vs, vz) = ops.quant_pack_rows(k, group, bits, True), ops.quant_pack_rows(v, group, bits, True)
    few = torch.arange(Lq, device=dev) % 2 == 0
    lim = torch.where(few, 32, Lk).int().contiguous()
    run = lambda: ops.fused_attn(q, *kq, vw, vs, vz, bits, bits, Lk, 1 / math.sqrt(D), kv_limit=lim)
    note('key waves, NaN behind the limit', D, bad, waves)
    want = run()
    vs[:, :, 40] = bad
    out = run()
    assert torch.equal(out[:, :, few], want[:, :, few])
    assert not bool(torch.isfinite(out[:, :, ~few]).all(-1).any())
