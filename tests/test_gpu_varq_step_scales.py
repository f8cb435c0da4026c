"""`scale` and `zp` of a step that one native call has quantized and cached are tensors of their own, as after quant() and cache(): dense, and
a caller's to change without changing the cache; what is dequantized of the step then follows them."""
import pytest
import torch

from gpu_util import note
from var_q_amd import VAR_Q
from var_q_amd.quant import fused_attention, fused_step

pytestmark = pytest.mark.gpu


class General(VAR_Q):
    pass


@pytest.mark.parametrize('method', ['G_TOKEN', 'G_TOKEN_HEAD', 'G_SCALE', 'G_HEAD'])
@pytest.mark.parametrize('layout', ['BLHc', 'BHLc'])
@pytest.mark.parametrize('symmetric', [True, False])
@pytest.mark.parametrize('B,H,c,n', [(1, 1, 64, 1), (2, 5, 64, 9), (3, 4, 128, 70)])
def test_changing_the_scale_of_a_step_leaves_the_cache(dev, method, layout, symmetric, B, H, c, n):
    note('step scales', method, layout, symmetric, B, H, c, n)
    g = torch.Generator().manual_seed(n)
    shape = (B, n, H, c) if layout == 'BLHc' else (B, H, n, c)
    pairs = [[cls(4, layout, method, symmetric=symmetric) for _ in range(2)] for cls in (VAR_Q, General)]
    for z in pairs[0] + pairs[1]:
        z.reserve_tokens(2 * n)
    for _ in range(2):      # (the second step is the native call's: the first makes the room)
        q, k, v = [torch.randn(*shape, generator=g).to(dev, torch.bfloat16) for _ in range(3)]
        for pair in pairs:
            fused_step(q, k, v, *pair, 0.125)
    for z in pairs[0]:
        assert z._window is not None, 'the step did not take the native call'
    before = fused_attention(q, *pairs[0], 0.125)
    kept = [(z.cached_scale.clone(), None if symmetric else z.cached_zp.clone()) for z in pairs[0]]
    for pair in pairs:
        for z in pair:
            for t in (z.scale,) if symmetric else (z.scale, z.zp):
                assert t.is_contiguous()
                t.view(-1).add_(3.0)
    for a, b, (s, zp) in zip(*pairs, kept):
        assert torch.equal(a.scale, b.scale) and (symmetric or torch.equal(a.zp, b.zp))
        assert torch.equal(a.cached_scale, s) and (symmetric or torch.equal(a.cached_zp, zp))
        assert torch.equal(a.dequant_current(), b.dequant_current()) and torch.equal(a.dequant_all(), b.dequant_all())
    assert torch.equal(fused_attention(q, *pairs[0], 0.125), before)
