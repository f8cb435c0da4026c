"""Steps whose groups take several launches (three, or workgroups that share the groups), in the native call of a step: it takes them, and leaves
codes, scales and zero-points of quant() and cache(), which a subclass goes through, bit for bit."""
from ctypes import c_int64

import pytest
import torch

from gpu_util import note
from var_q_amd import VAR_Q, _lib

pytestmark = pytest.mark.gpu


class General(VAR_Q):
    pass


MASK = {'G_SCALE': (0b1111, 0b1111), 'G_HEAD': (0b1011, 0b1101), 'G_TOKEN': (0b1101, 0b1011), 'G_TOKEN_HEAD': (0b1001, 0b1001)}


@pytest.mark.parametrize('two', [True, False])
@pytest.mark.parametrize('symmetric', [True, False])
@pytest.mark.parametrize('layout', ['BLHc', 'BHLc'])
@pytest.mark.parametrize('method,B,H,n,c,bits,dtype,shards', [
    ('G_SCALE', 1, 3, 700, 64, 8, torch.bfloat16, 0),        # one group
    ('G_SCALE', 2, 5, 331, 96, 4, torch.float32, 0),
    ('G_HEAD', 8, 30, 400, 64, 8, torch.float16, 0),         # a group per head, fewer than the finalizing workgroup has
    ('G_HEAD', 64, 16, 256, 64, 2, torch.float16, 2),
    ('G_TOKEN', 64, 16, 253, 64, 4, torch.float16, 2),       # a ragged number of groups, shared
    ('G_TOKEN', 64, 24, 601, 64, 8, torch.bfloat16, 0),
    ('G_TOKEN_HEAD', 64, 16, 259, 64, 8, torch.float16, 0),  # thousands of groups
])
def test_several_launches(dev, method, B, H, n, c, bits, dtype, shards, layout, symmetric, two):
    note('step of several launches', method, B, H, n, c, bits, dtype, layout, symmetric, two)
    shape = (B, n, H, c) if layout == 'BLHc' else (B, H, n, c)
    if two and symmetric and dtype == torch.float16:
        got = _lib.load().varq_quant_pack_shards((c_int64 * 4)(*shape), MASK[method][layout != 'BLHc'], 2, 2, bits, 0)
        assert got == 0 if shards == 0 else got >= shards
    first = list(shape)
    first[1 if layout == 'BLHc' else 2] = 2
    g = torch.Generator().manual_seed(n + bits)
    native, general = [[cls(bits, layout, method, symmetric=symmetric) for _ in range(1 + two)] for cls in (VAR_Q, General)]
    for z in native + general:
        z.reserve_tokens(n + 4)
    for i, s in enumerate((first, shape, first)):
        xs = [(torch.randn(*s, generator=g) * (1 + j) + j).to(dev, dtype) for j in range(1 + two)]
        taken = VAR_Q._step_fast_pair(*native, *xs) if two else native[0]._step_fast(xs[0])
        assert taken or i == 0
        for z, x in zip(general + ([] if taken else native), xs + xs):
            z.quant(x)
            z.cache()
        for a, b in zip(native, general):
            for name in ('quantized_item', 'scale', 'zp', 'cached_item', 'cached_scale', 'cached_zp'):
                p, q = getattr(a, name), getattr(b, name)
                assert (p is None) == (q is None) and (p is None or torch.equal(p, q)), (i, name)
