"""The kernel that widens K and V tile by tile into rows in LDS, at the edges of what its threads and tiles take: pieces of a row of
every width (2 to 16 bytes), one, two and many tiles with whole and ragged ends, workgroups of four and eight wavefronts and of one buffer,
scale groups of K and V that differ, and per-channel tables of up to 16 segments that begin inside tiles, with zero-points for both, one or
neither of K and V -- against the oracle's operands (the bars of test_gpu_attention.py and test_gpu_attention_channel.py)."""
import math

import pytest
import torch

import varq_oracle as O
from gpu_util import note
from test_gpu_attention import _compare, _exact_fp64
from test_gpu_attention_channel import ORACLE_BAR
from var_q_amd import ops

pytestmark = pytest.mark.gpu

SIZES = [(1, 1), (33, 63), (130, 64), (257, 65), (31, 128), (200, 129), (129, 321)]
GROUPS = [(64, 32, 64, 'fp16'), (64, 64, 64, 'bf16'), (128, 32, 64, 'bf16'), (128, 128, 128, 'bf16')]
# (300 pairs: workgroups of four wavefronts, at head dim 64 and up to 128 queries; 130 are on the other side of that line)
CASES = [(*g, B, H, *size) for size in SIZES for B, H in ((1, 3), (75, 4)) for g in GROUPS if B == 1 or (g[0] == 64 and size[0] <= 130)]


@pytest.mark.parametrize('D,gk,gv,dtype,B,H,Lq,Lk', CASES)
@pytest.mark.parametrize('bits', [2, 4, 8])
def test_groups(dev, bits, D, gk, gv, dtype, B, H, Lq, Lk):
    seed = bits + D + gk + Lq * 7 + Lk
    gen = torch.Generator().manual_seed(seed)
    dt, scale = torch.float16 if dtype == 'fp16' else torch.bfloat16, 1 / math.sqrt(D)
    k, v = (O.synth_kv((B, H, Lk, D), seed + i, 'normal').to(dt) for i in (1, 2))
    q = torch.randn(B, H, Lq, D, generator=gen).to(dt)
    asym = seed % 2 == 0
    kq, ks, kz = O.quant_groupwise(k, gk, bits, asym)
    vq, vs, vz = O.quant_groupwise(v, gv, bits, asym)
    kd, vd = O.dequant_groupwise(kq, ks, kz, gk), O.dequant_groupwise(vq, vs, vz, gv)
    to = lambda t: None if t is None else t.contiguous().to(dev)
    note('tiles, groups', bits, D, gk, gv, dtype, B, H, Lq, Lk, asym)
    out = ops.fused_attn(to(q), to(O.pack_last_dim(kq, bits)[0]), to(ks), to(kz), to(O.pack_last_dim(vq, bits)[0]), to(vs), to(vz), bits, bits, Lk, scale, splits=1)
    torch.cuda.synchronize()
    _compare(out[:1], O.attention_ref(q[:1], kd[:1], vd[:1], scale, dtype=dt), _exact_fp64(q[:1], kd[:1], vd[:1], scale, None, dev), 'tiles, groups')
    if B > 1:
        _compare(out[-1:], O.attention_ref(q[-1:], kd[-1:], vd[-1:], scale, dtype=dt), _exact_fp64(q[-1:], kd[-1:], vd[-1:], scale, None, dev), 'tiles, groups')


@pytest.mark.parametrize('ends', [(1,), (5, 64, 70), (1, 2, 40, 63, 64, 65, 66, 100, 127, 128, 129, 130, 190, 191, 192, 257)])
@pytest.mark.parametrize('zp', ['none', 'both', 'k', 'v'])
@pytest.mark.parametrize('D,B,H', [(64, 1, 3), (64, 75, 4), (128, 1, 3)])
@pytest.mark.parametrize('bits', [2, 4, 8])
def test_tables(dev, bits, D, B, H, zp, ends):
    seed, Lq, Lk, scale = bits + D + len(ends) + B, 70, ends[-1], 1 / math.sqrt(D)
    gen = torch.Generator().manual_seed(seed)
    half = 1 << (bits - 1)
    q = torch.randn(B, H, Lq, D, generator=gen).bfloat16()
    codes = [torch.randint(-half, half, (B, H, Lk, D), generator=gen, dtype=torch.int8) for _ in range(2)]
    scales = [torch.rand(len(ends), H, D, generator=gen) * 0.2 + 0.02 for _ in range(2)]
    zps = [torch.randint(-half, half, (len(ends), H, D), generator=gen).float() if zp in ('both', w) else None for w in 'kv']
    seg = torch.bucketize(torch.arange(Lk), torch.tensor(ends), right=True)
    at = lambda t: t[seg].permute(1, 0, 2)[None]      # [1,H,Lk,D]
    kd, vd = ((c.float() - (0 if z is None else at(z))) * at(s) for c, s, z in zip(codes, scales, zps))
    to = lambda t: None if t is None else t.contiguous().to(dev)
    kw, vw = (to(O.pack_last_dim(c, bits)[0]) for c in codes)
    note('tiles, tables', bits, D, B, H, zp, ends)
    out = ops.fused_attn_channel(to(q), kw, to(scales[0]), to(zps[0]), vw, to(scales[1]), to(zps[1]), bits, Lk, scale, seg_ends=list(ends), splits=1)
    torch.cuda.synchronize()
    for b in {0, B - 1}:
        s = slice(b, b + 1)
        _compare(out[s], O.attention_ref(q[s], kd[s], vd[s], scale), _exact_fp64(q[s], kd[s], vd[s], scale, None, dev), 'tiles, tables', oracle_bar=ORACLE_BAR)
