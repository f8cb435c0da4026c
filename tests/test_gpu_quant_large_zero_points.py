"""Zero-points beyond what the rounding trick of the general quantizer holds (|zp| > 2^21: values far from zero in a narrow range), beside groups
within it, in one launch and in several: codes, scales and zero-points of the oracle; and in the launch that dequantizes the cache as well: the
values of the separate calls."""
import pytest
import torch

import varq_oracle as O
from gpu_util import note
from var_q_amd import VAR_Q, ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('bits', [2, 4, 8])
@pytest.mark.parametrize('shape,dims', [((2, 3, 70, 64), (0, 2)), ((300, 4, 33, 64), (0, 2)), ((4, 70, 3, 64), (0, 1)), ((2, 5, 33, 32), (0, 3))])
def test_values_far_from_zero(dev, shape, dims, bits):
    gen = torch.Generator().manual_seed(bits)
    x = torch.randn(shape, generator=gen)
    # (values a few units in the last place around 2048 and -65536, and around 0)
    far = torch.tensor([0.0, 2048.0, -65536.0])[torch.arange(shape[1] if 2 in dims or 3 in dims else shape[2]) % 3]
    far = far.view(1, -1, 1, 1) if 2 in dims or 3 in dims else far.view(1, 1, -1, 1)
    x = x * torch.where(far == 0, 1.0, far.abs() * 2.0 ** -23) + far
    q, s, z = O.quant_reduce(x, dims, bits, True)
    assert float(z.abs().max()) > 2 ** 21 and float(z.abs().min()) < 2 ** 10
    note('large zero-points', shape, dims, bits)
    words, gs, gz = ops.quant_pack(x.to(dev), dims, bits, asym=True)
    torch.cuda.synchronize()
    assert torch.equal(gs.cpu().reshape(s.shape), s) and torch.equal(gz.cpu().reshape(z.shape), z)
    assert torch.equal(words.cpu(), O.pack_last_dim(q, bits)[0])


@pytest.mark.parametrize('bits', [2, 4, 8])
def test_step_and_cache(dev, bits):
    one, steps = VAR_Q(bits, 'BHLc', symmetric=False), VAR_Q(bits, 'BHLc', symmetric=False)
    gen = torch.Generator().manual_seed(bits)
    for n in (1, 5, 40, 300):
        x = (torch.randn(2, 3, n, 64, generator=gen) * 2.0 ** -7 + torch.tensor([0.0, 1.0, -65536.0]).view(1, 3, 1, 1)).to(dev)
        note('large zero-points, step', bits, n)
        steps.quant(x)
        steps.cache()
        assert torch.equal(one.use_var_q(x), steps.dequant_all(torch.float32)) and torch.equal(one.cached_item, steps.cached_item)
        assert torch.equal(one.cached_zp, steps.cached_zp) and float(one.cached_zp.abs().max()) > 2 ** 21


@pytest.mark.parametrize('bits', [2, 4, 8])
@pytest.mark.parametrize('shape', [(2, 4, 70, 64), (300, 4, 33, 64)])      # one launch; three
def test_quotients_up_to_the_largest_float(dev, shape, bits):
    """Constant groups, whose scale is eps: values over eps up to where a product with the reciprocal may pass the largest float and the
    quotient does not."""
    eps, largest = 1e-12, torch.finfo(torch.float32).max
    x = torch.tensor([1e13, -2.0 ** 79, 2.0 ** 81, -largest * eps * 0.99999]).view(1, 4, 1, 1).expand(shape).contiguous()
    q, s, z = O.quant_reduce(x, (0, 2), bits, True, eps)
    assert bool(torch.isfinite(z).all()) and float(z.abs().max()) > 2.0 ** 127
    note('quotients up to the largest float', shape, bits)
    words, gs, gz = ops.quant_pack(x.to(dev), (0, 2), bits, asym=True, eps=eps)
    assert torch.equal(gs.cpu().reshape(s.shape), s) and torch.equal(gz.cpu().reshape(z.shape), z)
    assert torch.equal(words.cpu(), O.pack_last_dim(q, bits)[0])
