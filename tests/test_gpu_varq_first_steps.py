"""The first step of a quantizer and steps that find its buffers full, for every rule that the native call of a step takes: it takes them too, with
and without the dequantized cache behind it, bit for bit what quant() and cache() (which a subclass goes through) leave."""
import pytest
import torch

from gpu_util import note
from var_q_amd import VAR_Q

pytestmark = pytest.mark.gpu


class General(VAR_Q):
    general = VAR_Q.quant

    def quant(self, item):
        return General.general(self, item)


@pytest.mark.parametrize('method', ['G_SCALE_HEAD_DIM', 'G_SCALE', 'G_HEAD', 'G_TOKEN', 'G_TOKEN_HEAD'])
@pytest.mark.parametrize('layout', ['BLHc', 'BHLc'])
@pytest.mark.parametrize('symmetric', [True, False])
@pytest.mark.parametrize('use', [None, torch.float32, torch.float16])
@pytest.mark.parametrize('steps', [(1, 1), (64, 1, 150), (70, 60)])      # room for 64 tokens at first: exactly full, and beyond
def test_first_and_growing_steps(dev, monkeypatch, method, layout, symmetric, use, steps):
    _steps(dev, monkeypatch, method, layout, symmetric, use, steps, 8, 64)


@pytest.mark.parametrize('method', ['G_SCALE_HEAD_DIM', 'G_SCALE', 'G_HEAD', 'G_TOKEN', 'G_TOKEN_HEAD'])
@pytest.mark.parametrize('layout', ['BLHc', 'BHLc'])
@pytest.mark.parametrize('use', [None, torch.bfloat16])
@pytest.mark.parametrize('bits,c', [(8, 24), (4, 40), (4, 128), (2, 48), (2, 128)])
def test_other_rows(dev, monkeypatch, method, layout, use, bits, c):
    _steps(dev, monkeypatch, method, layout, bits != 4, use, (1, 63, 1, 80), bits, c)


def _steps(dev, monkeypatch, method, layout, symmetric, use, steps, bits, c):
    note('first steps', method, layout, symmetric, use, steps, bits, c)
    d, g = 1 if layout == 'BLHc' else 2, torch.Generator().manual_seed(sum(steps))
    a, b = [cls(bits, layout, method, symmetric=symmetric) for cls in (VAR_Q, General)]
    with pytest.raises(RuntimeError):
        a.use_var_q(torch.empty((2, 0, 3, c) if d == 1 else (2, 3, 0, c), device=dev))
    assert a._pack_meta is None and a._c_item.buf is None

    def refuse(self, item):
        raise AssertionError('the general method of a quantizer that has a native step')
    monkeypatch.setattr(VAR_Q, 'quant', refuse)
    for n in steps:
        x = torch.randn(*((2, n, 3, c) if d == 1 else (2, 3, n, c)), generator=g).to(dev, torch.bfloat16)
        if use is None:
            assert a._step_fast(x)
            General.general(b, x)
            b.cache()
            got = want = None
        else:
            got, want = a.use_var_q(x, use), None
            if method == 'G_SCALE_HEAD_DIM':     # (a subclass has the native step of this rule as well)
                General.general(b, x)
                b.cache()
                want = b.dequant_all(use)
            else:
                want = b.use_var_q(x, use)
        for p, q in [(got, want)] + [(getattr(a, name), getattr(b, name)) for name in ('quantized_item', 'scale', 'zp', 'cached_item', 'cached_scale', 'cached_zp')]:
            assert (p is None) == (q is None) and (p is None or (p.shape == q.shape and torch.equal(p, q)))
    assert a._seg_ends == b._seg_ends and a._scale_shape == b._scale_shape and a._pack_meta == b._pack_meta
