"""A PackedKVCache is what its attributes say at each call: buffers, sizes and options that a caller sets after the
construction are those that append, attend and dequant use, and buffers that do not fit are refused."""
import pytest
import torch

import varq_oracle as O
from gpu_util import note
from var_q_amd import PackedKVCache
from var_q_amd._lib import VarqError

pytestmark = pytest.mark.gpu
BUFFERS = ('k_words', 'k_scale', 'k_zp', 'v_words', 'v_scale', 'v_zp')


def _step(dev, n, seed, B=2, H=4, D=64):
    gen = torch.Generator(device=dev).manual_seed(seed)
    return [torch.randn(B, H, n, D, device=dev, generator=gen).bfloat16() for _ in range(3)]


@pytest.mark.parametrize('bits', [4, [2, 8, 4, 8]])
def test_buffers_replaced_after_construction(dev, bits):
    """The buffers give way to larger ones (the cache grows), in a cache of one width and of three."""
    note('cache state: larger buffers', bits)
    cache, whole = PackedKVCache(2, 4, 20, 64, bits, 32, dev), PackedKVCache(2, 4, 90, 64, bits, 32, dev)
    (_, k0, v0), (q, k1, v1) = _step(dev, 17, 1), _step(dev, 70, 2)
    for c in (cache, whole):
        c.append(k0, v0)
    for cl in cache.classes:
        for name in BUFFERS:
            old = getattr(cl, name)
            new = torch.zeros(*old.shape[:2], 90, old.shape[3], dtype=old.dtype, device=dev)
            new[:, :, :20] = old
            setattr(cl, name, new)
            old.fill_(77)
    cache.Lmax = 90
    for c in (cache, whole):
        c.append(k1, v1)
    assert torch.equal(cache.attend(q, 0.125), whole.attend(q, 0.125))
    assert torch.equal(cache.dequant('k'), whole.dequant('k')) and torch.equal(cache.dequant('v'), whole.dequant('v'))
    qkv = torch.randn(2, 3, 3, 4, 64, device=dev, generator=torch.Generator(device=dev).manual_seed(3)).bfloat16()
    assert torch.equal(cache.append_from_qkv(qkv), whole.append_from_qkv(qkv))
    for (n, a), b in zip(cache.tensors().items(), whole.tensors().values()):
        assert torch.equal(a, b), n


@pytest.mark.parametrize('bits', [4, [2, 8, 4, 8]])
def test_options_set_after_construction(dev, bits):
    note('cache state: options', bits)
    cache = PackedKVCache(2, 4, 20, 64, bits, 32, dev)
    cache.eps, cache.symmetric = 0.5, True
    _, k, v = _step(dev, 9, 4)
    cache.append(k, v)
    per_head = [bits] * 4 if isinstance(bits, int) else bits
    for h, b in enumerate(per_head):
        codes, s, _ = O.quant_groupwise(k[:, h].cpu(), 32, b, False, eps=0.5)
        assert torch.equal(cache.dequant('k')[:, h].cpu(), O.dequant_groupwise(codes, s, None, 32))


@pytest.mark.parametrize('bits', [4, [2, 8, 4, 8]])
@pytest.mark.parametrize('change', ['short', 'row', 'zp', 'type', 'stride', 'cpu', 'slot'])
def test_buffers_that_do_not_fit_are_refused(dev, bits, change):
    note('cache state: refused', bits, change)
    cache = PackedKVCache(2, 4, 20, 64, bits, 32, dev)
    q, k, v = _step(dev, 20, 5)
    cl = cache.classes[-1]
    if change == 'short':
        cl.v_words = cl.v_words[:, :, :19].contiguous()
    elif change == 'row':
        cl.k_scale = torch.zeros(*cl.k_scale.shape[:3], 1, device=dev)
    elif change == 'zp':
        cl.k_zp = cl.k_zp[:1]
    elif change == 'type':
        cl.k_words = cl.k_words.float()
    elif change == 'stride':
        cl.v_scale = torch.zeros(2, len(cl.heads), 20, 4, device=dev)[..., ::2]
    elif change == 'cpu':
        cl.v_zp = cl.v_zp.cpu()
    else:
        cl.slot = cl.slot[:3].contiguous()
    for call in (lambda: cache.append(k, v), lambda: cache.append_from_qkv(torch.zeros(2, 20, 3, 4, 64, device=dev).bfloat16())):
        with pytest.raises((VarqError, AssertionError)):
            call()
    assert cache.len == 0
    if not isinstance(bits, int):
        cache.len = 20
        with pytest.raises((VarqError, AssertionError)):
            cache.attend(q, 0.125)
