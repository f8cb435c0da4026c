"""A cache with several bit-widths, all classes in one launch: the appended codes and scales are those of one
cache per class, and attention that of one launch per class -- bit for bit where the keys are not shared
out, to rounding where they are -- at the edges of the launches: one head of a class, two classes, one
token, steps shorter and longer than the head count, K and V of different dtypes, few queries over
many keys (their own kernel), queries enough for the expanded tiles, key limits, tokens-first results."""
import pytest
import torch

from gpu_util import note
from var_q_amd import PackedKVCache, ops

pytestmark = pytest.mark.gpu


def _per_class(cache, q, scale, limit, splits):
    out = torch.zeros_like(q)
    for c in cache.classes:
        z = (None, None) if cache.symmetric else (c.k_zp, c.v_zp)
        ops.fused_attn(q, c.k_words, c.k_scale, z[0], c.v_words, c.v_scale, z[1], c.bits, c.bits, cache.len, scale,
                       kv_limit=limit, head_map=c.head_map, out=out, splits=splits)
    return out


@pytest.mark.parametrize('B,bits,D,group,steps,dtypes,layout,symmetric', [
    (1, '28', 128, 128, (1, 3, 64), 'bb', 'BHLc', False),
    (2, '4284848', 128, 64, (5, 33, 1300), 'bb', 'BLHc', False),
    (3, '244442', 64, 32, (7, 100, 129), 'hh', 'BHLc', True),
    (33, '82488848', 64, 64, (1, 40, 90), 'hh', 'BLHc', False),       # more pairs than compute units
    (1, '848', 128, 32, (2, 1500, 30), 'fb', 'BHLc', True),
    (2, '2842', 128, 128, (6, 1100, 17), 'bb', 'BHLc', False),        # ends in few queries over many keys
    (5, '82488848', 64, 64, (600, 1600), 'bb', 'BLHc', False),        # ends in expanded tiles
    (4, '24424424', 128, 16, (9, 20), 'bb', 'BHLc', False),           # groups that only the launches per class know
])
def test_classes_in_one_launch(dev, B, bits, D, group, steps, dtypes, layout, symmetric):
    types = {'b': torch.bfloat16, 'h': torch.float16, 'f': torch.float32}
    kt, vt = types[dtypes[0]], types[dtypes[1]]
    H, L = len(bits), sum(steps)
    per_head = [int(b) for b in bits]
    gen = torch.Generator().manual_seed(L)
    cache = PackedKVCache(B, H, L + 3, D, per_head, group, dev, symmetric=symmetric)
    single = {b: PackedKVCache(B, per_head.count(b), L + 3, D, b, group, dev, symmetric=symmetric) for b in sorted(set(per_head))}
    pick = {b: [h for h in range(H) if per_head[h] == b] for b in single}
    hd = 1 if layout == 'BHLc' else 2
    for n in steps:
        shape = (B, H, n, D) if layout == 'BHLc' else (B, n, H, D)
        k, v = torch.randn(*shape, generator=gen).to(kt).to(dev), (torch.randn(*shape, generator=gen) * 3 + 1).to(vt).to(dev)
        note('classes', B, bits, D, group, n, dtypes, layout)
        cache.append(k, v, layout)
        for b, one in single.items():
            idx = torch.tensor(pick[b], device=dev)
            one.append(k.index_select(hd, idx), v.index_select(hd, idx), layout)
    torch.cuda.synchronize()
    got = cache.tensors()
    for one in single.values():
        for name, t in one.tensors().items():
            assert torch.equal(got[name], t), name
    if group < 32:
        return
    n, scale = steps[-1], 0.08
    q = torch.randn(B, H, n, D, generator=gen).to(torch.float16 if dtypes == 'hh' else torch.bfloat16).to(dev)
    for limit in (None, torch.randint(0, L + 1, (n,), generator=gen).int().to(dev)):
        want = _per_class(cache, q, scale, limit, 1)
        cache.splits = 1
        a = cache.attend(q, scale, kv_limit=limit)
        cache.splits = 0
        b = cache.attend(q, scale, kv_limit=limit, out_layout='BLHc')
        torch.cuda.synchronize()
        if n != 1600:   # (there the cache as a whole takes the expanded tiles, a class by itself does not)
            assert torch.equal(a, want)
        assert b.shape == (B, n, H, D)
        torch.testing.assert_close(a.float(), want.float(), rtol=2e-2, atol=2e-2)
        torch.testing.assert_close(b.transpose(1, 2).float(), want.float(), rtol=2e-2, atol=2e-2)


@pytest.mark.parametrize('D,group,n', [(128, 64, 1), (128, 128, 37), (64, 32, 130)])
def test_classes_from_qkv(dev, D, group, n):
    B, bits, start = 2, [2, 8, 4, 4, 8], 5
    H = len(bits)
    gen = torch.Generator().manual_seed(n)
    qkv = torch.randn(B, n, 3, H, D, generator=gen).bfloat16().to(dev)
    mul = (torch.rand(H, generator=gen) + 1).to(dev)
    cs, sn = (torch.randn(start + n, D // 2, generator=gen).to(dev) for _ in range(2))
    note('classes from qkv', D, group, n)
    cache = PackedKVCache(B, H, start + n, D, bits, group, dev)
    cache.len = start
    q = cache.append_from_qkv(qkv, mul, l2norm=True, rope=(cs, sn))
    for b in sorted(set(bits)):
        idx = torch.tensor([h for h in range(H) if bits[h] == b], device=dev)
        one = PackedKVCache(B, len(idx), start + n, D, b, group, dev)
        one.len = start
        q1 = one.append_from_qkv(qkv.index_select(3, idx), mul[idx].contiguous(), l2norm=True, rope=(cs, sn))
        torch.cuda.synchronize()
        assert torch.equal(q.index_select(1, idx), q1)
        for name, t in one.tensors().items():
            assert torch.equal(cache.tensors()[name], t), name
