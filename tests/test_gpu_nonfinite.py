"""Infinities, NaN and the types' lowest values: the one-launch quantizer gives what the three launches give, bit for bit, the
one-call step what the three calls give, and the attention that expands K and V first is finite where the kernel that widens
per workgroup is."""
import math

import pytest
import torch

from gpu_util import note
from var_q_amd import VAR_Q, ops

pytestmark = pytest.mark.gpu
INF, NAN = math.inf, math.nan


def _spoil(x, tokens, what):
    """Puts `what` into some of the groups of x; tokens: its dim of the tokens."""
    x = x.clone()
    last, lowest = x.shape[tokens] - 1, torch.finfo(x.dtype).min
    at = lambda t: [slice(None)] * tokens + [t]
    values = {'nan': [NAN], 'inf': [INF], '-inf': [-INF], 'both': [INF, -INF], 'inf and nan': [INF, NAN], 'lowest': [lowest], 'range': [lowest, -lowest]}
    if what in values:
        for i, v in enumerate(values[what]):
            x[tuple(at(min(i, last)))][..., 1::3] = v
    else:     # whole groups
        x[..., 2::5] = {'all nan': NAN, 'all inf': INF, 'all -inf': -INF, 'all lowest': lowest}[what]
    return x


def _bits(t):
    """The bits, NaN as one value."""
    t = torch.where(torch.isnan(t), torch.full_like(t, NAN), t)
    return t.view(torch.int32 if t.dtype == torch.float32 else torch.int16)


WHAT = ['nan', 'inf', '-inf', 'both', 'inf and nan', 'lowest', 'range', 'all nan', 'all inf', 'all -inf', 'all lowest']


@pytest.mark.parametrize('what', WHAT)
@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize('shape,dims', [((2, 3, 300, 64), (0, 2)), ((4, 70, 3, 64), (0, 1)), ((2, 5, 33, 32), (0, 3)), ((2, 3, 40, 48), (0, 2, 3))])
def test_one_launch_and_three(dev, shape, dims, dtype, what):
    """The batch often enough behind itself leaves every group what it is and makes it too long for one launch (8192 rows), or
    the tensor too large (48 MiB)."""
    x = _spoil(torch.randn(*shape, generator=torch.Generator().manual_seed(7)).to(dtype).to(dev), 1 if dims == (0, 1) else 2, what)
    rows = math.prod(shape[d] for d in dims if d != 3)
    times = max(8192 // rows + 1, (48 << 20) // (x.numel() * x.element_size()) + 1 if 3 in dims else 0)
    for bits, asym in ((8, False), (8, True), (4, True), (2, False), (2, True)):
        note('non-finite', shape, dims, dtype, what, bits, asym)
        q1, s1, z1 = ops.quant_pack(x, dims, bits, asym=asym)
        q3, s3, z3 = ops.quant_pack(x.repeat(times, 1, 1, 1), dims, bits, asym=asym)
        assert torch.equal(_bits(s1), _bits(s3)) and (not asym or torch.equal(_bits(z1), _bits(z3)))
        assert torch.equal(q1, q3[:shape[0]])


@pytest.mark.parametrize('what', WHAT)
@pytest.mark.parametrize('fmt', ['BHLc', 'BLHc'])
@pytest.mark.parametrize('bits,symmetric', [(8, True), (4, False), (2, False)])
def test_one_call_and_three(dev, fmt, bits, symmetric, what):
    gen = torch.Generator().manual_seed(bits)
    one, three = (VAR_Q(bits, fmt, symmetric=symmetric) for _ in range(2))
    for i, n in enumerate((1, 3, 70, 200)):
        x = torch.randn(*((2, 3, n, 64) if fmt == 'BHLc' else (2, n, 3, 64)), generator=gen).to((torch.float32, torch.bfloat16, torch.float16)[i % 3]).to(dev)
        if i != 1:
            x = _spoil(x, 2 if fmt == 'BHLc' else 1, what)
        note('non-finite step', fmt, bits, what, n)
        three.quant(x)
        three.cache()
        for out in (torch.float32, torch.bfloat16, torch.float16)[:3 if i == 3 else 1]:
            want = three.dequant_all(out)
            got = one.use_var_q(x, out) if out == torch.float32 else one.dequant_all(out)
            assert torch.equal(_bits(got), _bits(want))
        assert torch.equal(one.cached_item, three.cached_item) and torch.equal(_bits(one.cached_scale), _bits(three.cached_scale))


@pytest.mark.parametrize('D,group,H,dtype', [(128, 128, 20, 'bf16'), (64, 32, 22, 'fp16')])
@pytest.mark.parametrize('side,value', [('k', NAN), ('k', INF), ('v', NAN), ('v', INF), ('q', NAN), ('q', INF), ('k', 1e30)])
def test_expanding_attention(dev, D, group, H, dtype, side, value):
    """One key (scales of K or V) or some queries of some heads are spoilt, in the first, a middle and the last tile.  Blocks
    that a workgroup has whole and blocks that several share."""
    dt = torch.float16 if dtype == 'fp16' else torch.bfloat16
    B, Lq, Lk = 2, 1700, 2100
    gen = torch.Generator(device=dev).manual_seed(5)
    q = torch.randn(B, H, Lq, D, device=dev, generator=gen).to(dt)
    kq, vq = ([t.clone() for t in ops.quant_pack_rows(torch.randn(B, H, Lk, D, device=dev, generator=gen).bfloat16(), group, 4, True)] for _ in range(2))
    spoilt = {(0, 0): 0, (0, 3): 1000, (1, 1): Lk - 1, (1, H - 1): 70}
    for (b, h), key in spoilt.items():
        if side == 'q':
            q[b, h, 5:1700:40] = value
        else:
            (kq if side == 'k' else vq)[1][b, h, key] = value
    note('non-finite attention', D, side, value)
    run = lambda **kw: ops.fused_attn(q, *kq, *vq, 4, 4, Lk, 1 / math.sqrt(D), **kw)
    other = run(splits=2)
    fine = torch.isfinite(run(splits=1))
    for out in (run(), run(kv_limit=torch.full((Lq,), Lk, dtype=torch.int32, device=dev))):
        assert torch.equal(torch.isfinite(out), fine)
    whole = [i for i in range(B * H) if (i // H, i % H) not in spoilt]
    assert bool(fine.flatten(0, 1)[whole].all())
    if math.isnan(value):
        want = torch.ones_like(fine)
        for b, h in spoilt:
            if side == 'q':
                want[b, h, 5:1700:40] = False
            else:
                want[b, h] = False
        assert torch.equal(fine, want) and torch.equal(torch.isfinite(other), want)


@pytest.mark.parametrize('Lq,Lk,splits', [(16, 3000, 0), (50, 2100, 0), (300, 700, 3), (600, 700, 8), (2000, 700, 2)])
@pytest.mark.parametrize('value', [NAN, INF])
def test_shares_of_the_keys(dev, Lq, Lk, splits, value):
    """A NaN in one share of the keys is one in the result, as without shares; both ways of putting shares together, and the
    wavefronts of the kernel for few queries."""
    B, H, D = 2, 5, 128
    gen = torch.Generator(device=dev).manual_seed(8)
    q = torch.randn(B, H, Lq, D, device=dev, generator=gen).bfloat16()
    kq, vq = ([t.clone() for t in ops.quant_pack_rows(torch.randn(B, H, Lk, D, device=dev, generator=gen).bfloat16(), 128, 4, True)] for _ in range(2))
    kq[1][0, 1, 650] = value
    kq[1][1, 4, 0] = value
    note('non-finite shares', Lq, Lk, splits, value)
    run = lambda n: torch.isfinite(ops.fused_attn(q, *kq, *vq, 4, 4, Lk, 0.09, splits=n))
    want = torch.ones(B, H, Lq, D, dtype=torch.bool, device=dev)
    want[0, 1] = want[1, 4] = False
    assert torch.equal(run(1), want) and torch.equal(run(splits), want)


def test_keys_behind_the_limit_may_hold_anything_in_k(dev):
    B, H, L, D = 1, 27, 2100, 128
    gen = torch.Generator(device=dev).manual_seed(6)
    q = torch.randn(B, H, L, D, device=dev, generator=gen).bfloat16()
    kq, vq = ([t.clone() for t in ops.quant_pack_rows(torch.randn(B, H, L, D, device=dev, generator=gen).bfloat16(), 128, 4, True)] for _ in range(2))
    limit = torch.full((L,), 1025, dtype=torch.int32, device=dev)
    run = lambda: ops.fused_attn(q, *kq, *vq, 4, 4, L, 0.09, kv_limit=limit)
    note('non-finite keys behind the limit')
    want = run()
    kq[1][:, :, 1025:] = NAN
    assert bool(torch.isfinite(want).all()) and torch.equal(run(), want)
