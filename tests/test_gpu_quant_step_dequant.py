"""`use_var_q` of the shipped rule goes through one library call, and for small steps one launch, that quantizes the
step and dequantizes the cache; `quant` + `cache` + `dequant_all` take a launch for each.  Same codes, tables and
values, bit for bit, at every step: one row per workgroup to several, none to many earlier tokens, steps too large
for one launch, and a quantizer that changes between the two ways."""
import pytest
import torch

from gpu_util import note
from var_q_amd import VAR_Q

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('fmt', ['BHLc', 'BLHc'])
@pytest.mark.parametrize('bits,c', [(2, 16), (2, 128), (4, 8), (4, 64), (8, 64), (8, 72), (8, 520)])
@pytest.mark.parametrize('B,H,steps', [(1, 1, (1, 1, 3)), (3, 5, (1, 4, 37, 300, 2)), (64, 6, (2, 1, 40, 200)), (2, 16, (9, 6200, 1, 129))])
@pytest.mark.parametrize('symmetric', [True, False])
def test_equals_the_three_calls(dev, fmt, bits, c, B, H, steps, symmetric):
    if B * H * c * sum(steps) > 3e7:
        pytest.skip('large')
    gen = torch.Generator(device=dev).manual_seed(bits * c + B)
    dts = (torch.float32, torch.bfloat16, torch.float16)
    one, three = (VAR_Q(bits, fmt, 'G_SCALE_HEAD_DIM', symmetric=symmetric) for _ in range(2))
    for i, n in enumerate(steps):
        dt, out = dts[(i + c) % 3], dts[(i + bits // 2) % 3]
        x = (torch.randn(*((B, H, n, c) if fmt == 'BHLc' else (B, n, H, c)), device=dev, generator=gen) * 3 + 0.5).to(dt)
        note('use_var_q', fmt, bits, B, H, c, n, dt, out, symmetric)
        three.quant(x)
        three.cache()
        want = three.dequant_all(out)
        if i == 2:   # (this step the other way)
            one.quant(x)
            one.cache()
            got = one.dequant_all(out)
        else:
            got = one.use_var_q(x, out)
        assert got.dtype == out and got.is_contiguous() and torch.equal(got, want)
        assert torch.equal(one.cached_item, three.cached_item) and torch.equal(one.scale, three.scale)
        assert torch.equal(one.quantized_item, three.quantized_item)
        assert symmetric or torch.equal(one.zp, three.zp)
    assert torch.equal(one.cached_scale, three.cached_scale)
