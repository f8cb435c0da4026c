"""Key limits under which the wavefronts (32 queries) and the query tiles (256) of a (batch, head) pair end at
different keys: none at all, one, the edges of a 32-key block and of a 64-key tile, all, rising and falling.
The pairs do not fill the eight classes that the workgroups are dealt out to."""
import math

import pytest
import torch

import varq_oracle as O
from gpu_util import note
from test_gpu_attention import _compare, _quantize
from var_q_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('exact_codes', [False, True])
@pytest.mark.parametrize('layout', ['BHLc', 'BLHc'])
@pytest.mark.parametrize('splits', [0, 3])
@pytest.mark.parametrize('D,bits,group,B,H,Lq,Lk,order', [
    (64, 4, 32, 3, 7, 680, 680, 'rising'),      # three query tiles
    (64, 8, 64, 3, 3, 1025, 300, 'rising'),     # five, the last with one query
    (64, 2, 64, 2, 5, 257, 129, 'falling'),
    (128, 4, 128, 3, 3, 513, 450, 'rising'),
    (128, 4, 128, 1, 5, 300, 257, 'falling'),
    (64, 4, 64, 30, 9, 100, 200, 'rising'),     # workgroups of four wavefronts
])
def test_wavefronts_end_at_different_keys(dev, D, bits, group, B, H, Lq, Lk, order, splits, layout, exact_codes):
    if exact_codes and D != 128:
        pytest.skip('exact codes exist at head dim 128')
    gen = torch.Generator().manual_seed(Lq + Lk + D)
    k, v, q = (torch.randn(B, H, n, D, generator=gen).bfloat16() for n in (Lk, Lk, Lq))
    steps = [0, 1, 31, 32, 33, 63, 64, 65, 97, 128, Lk - 1, Lk]
    if order == 'falling':
        steps = steps[::-1]
    lim = torch.tensor(steps, dtype=torch.int32)[torch.arange(Lq) * len(steps) // Lq]
    (kw, ks, kz, kd), (vw, vs, vz, vd) = _quantize(k, group, bits), _quantize(v, group, bits)
    scale = 1 / math.sqrt(D)
    put = (lambda t: t.transpose(1, 2).contiguous().to(dev)) if layout == 'BLHc' else (lambda t: t.to(dev))
    note('key limits by wavefront', (D, bits, group, B, H, Lq, Lk), order, splits, layout, exact_codes)
    out = ops.fused_attn(*map(put, (q, kw, ks, kz, vw, vs, vz)), bits, bits, Lk, scale, kv_limit=lim.to(dev), splits=splits, layout=layout,
                         exact_codes=exact_codes)
    out = (out.transpose(1, 2) if layout == 'BLHc' else out).cpu()
    seen = lim > 0
    assert bool((out[:, :, ~seen] == 0).all())
    bias = torch.zeros(Lq, Lk).masked_fill(torch.arange(Lk)[None] >= lim[:, None], -math.inf)[seen]
    some = slice(0, 3) if B > 3 else slice(None)
    ref = O.attention_ref(q[some, :, seen], kd[some], vd[some], scale, bias)
    _compare(out[some, :, seen], ref, O.attention_exact(q[some, :, seen].float(), kd[some], vd[some], scale, bias), 'limits', exact_codes=exact_codes)
