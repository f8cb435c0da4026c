"""Stepwise caches with more than 65535 (batch, head) pairs: each of the two dims may be that large (the limit of a
launch grid's dim), as for the general dequantization.  One workgroup or two of a pair, the pair's head in the table."""
import pytest
import torch

import varq_oracle as O
from gpu_util import note
from var_q_amd import VAR_Q
from var_q_amd._lib import VarqError

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('B,H,c,steps', [(4096, 17, 16, (1, 1, 2)), (9000, 8, 8, (1, 3)), (1, 65535, 8, (1, 2)), (33, 2000, 128, (1, 70))])
@pytest.mark.parametrize('symmetric', [True, False])
def test_many_pairs(dev, B, H, c, steps, symmetric):
    note('dequant_steps pairs', B, H, c, steps, symmetric)
    gen = torch.Generator().manual_seed(B + H)
    z, two, want = VAR_Q(8, 'BHLc', symmetric=symmetric), VAR_Q(8, 'BHLc', symmetric=symmetric), []
    for i, n in enumerate(steps):
        x = torch.randn(B, H, n, c, generator=gen) * (i + 1) + 0.3
        codes, s, zp = O.quant_reduce(x, (0, 2), 8, not symmetric)
        want.append(O.dequant_sym(codes, s) if symmetric else O.dequant_asym(codes, s, zp))
        two.quant(x.to(dev))
        two.cache()
        got = z.use_var_q(x.to(dev))
        assert torch.equal(got.cpu(), torch.cat(want, 2)) and torch.equal(two.dequant_all(), got)


def test_a_dim_beyond_the_grid_is_refused_before_the_step_is_cached(dev):
    z = VAR_Q(8, 'BLHc')
    note('dequant_steps: 65536 batch entries')
    with pytest.raises(VarqError):
        z.use_var_q(torch.randn(65536, 1, 2, 8, device=dev))
    assert z._c_item.len == 0 and not z._seg_ends


def test_counts_beyond_31_bits_take_the_general_launch():
    z = VAR_Q(8, 'BLHc')
    assert z._steps_fit(65535, 32767, 8) and not z._steps_fit(65535, 32769, 8) and z._steps_fit((1 << 31) - 2049, 1, 8)
    z.qkv_format = 'BHLc'
    assert z._steps_fit(65535, 1 << 20, 8) and not z._steps_fit((1 << 31) - 2048, 1, 8)
