"""The step of a quantizer in one native call, with codes and scales written where the cache keeps them, against quant() and cache(),
which a subclass goes through: the same codes, scales, zero-points, attention and dequantized cache, bit for bit, for every rule that the
call takes, in both layouts, over steps of one token and of many, growing buffers, and steps too large for the one launch."""
import pytest
import torch

from gpu_util import note
from var_q_amd import VAR_Q
from var_q_amd.quant import fused_step

pytestmark = pytest.mark.gpu


class General(VAR_Q):
    pass


def _same(a, b):
    assert (a is None) == (b is None)
    assert a is None or (a.shape == b.shape and a.dtype == b.dtype and torch.equal(a, b))


@pytest.mark.parametrize('method', ['G_TOKEN', 'G_TOKEN_HEAD', 'G_SCALE', 'G_HEAD'])
@pytest.mark.parametrize('layout', ['BLHc', 'BHLc'])
@pytest.mark.parametrize('B,H,c,bits,symmetric,dtype,steps', [
    (1, 1, 64, 8, True, torch.float16, (1, 1, 2, 3)),
    (2, 5, 64, 4, False, torch.float16, (1, 4, 9, 25, 36)),
    (3, 3, 128, 2, False, torch.bfloat16, (2, 33, 65, 7)),             # the buffers of 64 tokens grow
    (2, 7, 128, 8, False, torch.float32, (5, 300, 1)),
    (2, 2, 24, 8, True, torch.bfloat16, (1, 17, 3)),                   # (no attention over 24 channels)
    (4, 16, 128, 4, True, torch.bfloat16, (3, 2, 2100, 1)),            # a step that takes several launches between two that take one
    (16, 16, 64, 8, True, torch.float16, (3, 600, 1)),                 # 37 MiB of K and V in one launch under the rules of whole rows
])
def test_same_state_as_the_general_calls(dev, method, layout, B, H, c, bits, symmetric, dtype, steps):
    g = torch.Generator().manual_seed(B * 1000 + H * 10 + bits)
    made = [cls(bits, layout, method, symmetric=symmetric) for cls in (VAR_Q, General) for _ in range(2)]
    alone = [cls(bits, layout, method, symmetric=symmetric) for cls in (VAR_Q, General)]
    native, general = made[:2], made[2:]
    for n in steps:
        shape = (B, n, H, c) if layout == 'BLHc' else (B, H, n, c)
        k, v = [(torch.randn(*shape, generator=g) * (1 + i)).to(dev, dtype) for i in range(2)]
        note('step', method, layout, shape, bits, symmetric, dtype)
        if c == 24:
            for pair in (native, general):
                if not VAR_Q._step_fast_pair(*pair, k, v):
                    for quantizer, x in zip(pair, (k, v)):
                        quantizer.quant(x)
                        quantizer.cache()
        else:
            _same(*[fused_step(k * 0.1, k, v, *pair, 0.125) for pair in (native, general)])
        _same(*[quantizer.use_var_q(v, torch.bfloat16) for quantizer in alone])
        for a, b in list(zip(native, general)) + [alone]:
            for name in ('quantized_item', 'scale', 'zp', 'cached_item', 'cached_scale', 'cached_zp'):
                _same(getattr(a, name), getattr(b, name))
            assert a._seg_ends == b._seg_ends and a._scale_shape == b._scale_shape and a._pack_meta == b._pack_meta


@pytest.mark.parametrize('layout', ['BLHc', 'BHLc'])
@pytest.mark.parametrize('symmetric', [True, False])
@pytest.mark.parametrize('c', [4, 12, 20, 100])
def test_channels_that_are_no_whole_octets(dev, layout, symmetric, c):
    """The shipped rule at 8 bits takes whole words of channels in one call: alone, both tensors of a step, and with the cache
    dequantized; the state is that of quant() and cache(), past the steps that the tables hold too."""
    g = torch.Generator().manual_seed(c)
    make = lambda: VAR_Q(8, layout, symmetric=symmetric)
    alone, pair, used, general = make(), [make(), make()], make(), [make(), make()]
    for i in range(18):
        n = (3, 1, 70)[i % 3]
        shape = (2, n, 3, c) if layout == 'BLHc' else (2, 3, n, c)
        k, v = [torch.randn(*shape, generator=g).to(dev) for _ in range(2)]
        note('step of', c, 'channels', layout, symmetric, i)
        took = [alone._step_fast(k), VAR_Q._step_fast_pair(*pair, k, v)]
        assert took == [i < 16] * 2
        for z, x in zip([alone, *pair][0 if i >= 16 else 3:] + general, (k, k, v, k, v)[0 if i >= 16 else 3:]):
            z.quant(x)
            z.cache()
        _same(used.use_var_q(k), general[0].dequant_all())
        for a, b in ((alone, general[0]), (pair[0], general[0]), (pair[1], general[1]), (used, general[0])):
            for name in ('quantized_item', 'scale', 'zp', 'cached_item', 'cached_scale', 'cached_zp'):
                _same(getattr(a, name), getattr(b, name))
            _same(a.dequant_current(), b.dequant_current())
            _same(a.dequant_all(), b.dequant_all())
            assert a._seg_ends == b._seg_ends and a._scale_shape == b._scale_shape and a._pack_meta == b._pack_meta
